// float32 values in the three products.
//
// The reference's launchers pass whatever dtype the tensors have to kernels that accumulate in fp32
// (stk/backend/triton_kernels.py:250, 306, 358; ACC_TYPE :248): float32 operands are legal there.  The 16-bit
// tile engine (gemm_core.h) does not take them, so stk_sdd / stk_dsd / stk_dds hand STK_F32 problems to the
// kernels here, all on v_mfma_f32_32x32x2_f32 (256 FLOP per cycle and compute unit, a sixteenth of the bf16 rate: it is
// the matrix pipe that bounds them, and what is left to choose is how many compute units get work).  Two sets:
//   Fast     operands with a unit stride, 16-byte aligned, extents that are whole tiles: operand tiles go from memory
//            to LDS without passing through registers, in a ring of two to four K-tiles of 32; output tiles of
//            128x128, 64x64 or 32x32 (fast_tile).
//   generic  any strides and ragged dense extents: one BLK x BLK tile per workgroup of four wavefronts, 16 k at a time
//            through registers, predicated.
// The walks are those of the 16-bit kernels.  A plan, a workspace or a block order are ignored: results never depend
// on them.
#include "common.h"
#include "gemm_core.h"

namespace stk {

namespace f32 {

constexpr int kKT = 16;        // k per staged tile
constexpr int kThreads = 256;  // 2 x 2 wavefronts
constexpr int kPad = 4;        // floats between LDS rows: the staging writes of a K-major tile spread over the banks

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One operand of a K-tile: EXT (m or n extent) x kKT elements at p[mn * s_mn + k * s_k], mn < valid, held by a
// thread as EXT * kKT / kThreads values.  K-major (s_k == 1): consecutive threads run along k; otherwise along mn.
template <int EXT>
struct Staged {
  static constexpr int kPer = EXT * kKT / kThreads;  // 8 (EXT 128) or 4 (EXT 64)
  float v[kPer];
  __device__ __forceinline__ static void place(int i, int tid, bool kmajor, int& mn, int& k) {
    const int e = i * kThreads + tid;
    if (kmajor) mn = e / kKT, k = e % kKT;
    else mn = e % EXT, k = e / EXT;
  }
  __device__ __forceinline__ void load(const float* p, int64_t s_mn, int64_t s_k, int valid, int tid) {
    const bool kmajor = s_k == 1;
#pragma unroll
    for (int i = 0; i < kPer; i++) {
      int mn, k;
      place(i, tid, kmajor, mn, k);
      v[i] = mn < valid ? p[mn * s_mn + k * s_k] : 0.f;
    }
  }
  __device__ __forceinline__ void store(float* lds, int64_t s_k, int tid) const {
    const bool kmajor = s_k == 1;
#pragma unroll
    for (int i = 0; i < kPer; i++) {
      int mn, k;
      place(i, tid, kmajor, mn, k);
      lds[k * (EXT + kPad) + mn] = v[i];
    }
  }
};

template <int BLK>
struct Tile {
  static constexpr int kW = BLK / 64;  // 32x32 MFMA tiles per wavefront in each direction (wave tile BLK/2 x BLK/2)
  static constexpr int kLdsFloats = 2 * kKT * (BLK + kPad);
  f32x16_t acc[kW][kW];

  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < kW; i++)
#pragma unroll
      for (int j = 0; j < kW; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
  }

  // acc += A [BLK x klen] * B [klen x BLK]; A element (m, k) at a[m * a_sm + k * a_sk], B element (k, n) at
  // b[k * b_sk + n * b_sn]; rows >= m_valid of A and columns >= n_valid of B count as zero.  klen is a multiple of kKT.
  __device__ __forceinline__ void accumulate(const float* a, int64_t a_sm, int64_t a_sk, int m_valid,
                                             const float* b, int64_t b_sk, int64_t b_sn, int n_valid, int klen, float* lds) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = (wave & 1) * (BLK / 2), n0 = (wave >> 1) * (BLK / 2);
    float* as = lds;
    float* bs = lds + kKT * (BLK + kPad);
    Staged<BLK> ra, rb;
    ra.load(a, a_sm, a_sk, m_valid, tid);
    rb.load(b, b_sn, b_sk, n_valid, tid);
    for (int k0 = 0; k0 < klen; k0 += kKT) {
      __syncthreads();  // the previous K-tile has been read by every wavefront
      ra.store(as, a_sk, tid);
      rb.store(bs, b_sk, tid);
      __syncthreads();
      if (k0 + kKT < klen) {
        ra.load(a + (int64_t)(k0 + kKT) * a_sk, a_sm, a_sk, m_valid, tid);
        rb.load(b + (int64_t)(k0 + kKT) * b_sk, b_sn, b_sk, n_valid, tid);
      }
#pragma unroll
      for (int ks = 0; ks < kKT; ks += 2) {
        // lane l: element (m or n = l % 32, k = ks + l / 32) of each 32-wide strip
        const int k = ks + (lane >> 5);
        float fa[kW], fb[kW];
#pragma unroll
        for (int i = 0; i < kW; i++) fa[i] = as[k * (BLK + kPad) + m0 + 32 * i + (lane & 31)];
#pragma unroll
        for (int j = 0; j < kW; j++) fb[j] = bs[k * (BLK + kPad) + n0 + 32 * j + (lane & 31)];
        // operands swapped, as in the 16-bit engine: a lane then owns four consecutive columns of one output row
#pragma unroll
        for (int i = 0; i < kW; i++)
#pragma unroll
          for (int j = 0; j < kW; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j], fa[i], acc[i][j], 0, 0, 0);
      }
    }
  }

  // out[m * ldc + n] = act(acc) (* mul[m * ldc + n]) for m < m_valid, n < n_valid; out points at the tile's corner.
  // Lane l holds in acc[i][j][4 g + q] the element (m = 32 i + l % 32, n = 32 j + 8 g + 4 (l / 32) + q) of its wave tile.
  __device__ __forceinline__ void store(float* out, int64_t ldc, int m_valid, int n_valid, int activation, const float* mul) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = (wave & 1) * (BLK / 2), n0 = (wave >> 1) * (BLK / 2);
    const bool vector = (ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(out) & 15u) == 0) &&
                        (!mul || (reinterpret_cast<uintptr_t>(mul) & 15u) == 0);
#pragma unroll
    for (int i = 0; i < kW; i++)
#pragma unroll
      for (int j = 0; j < kW; j++) {
        if (activation != kNoActivation) activate_all(acc[i][j], activation);
        const int m = m0 + 32 * i + (lane & 31);
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int n = n0 + 32 * j + 8 * g + 4 * (lane >> 5);
          if (m >= m_valid || n >= n_valid) continue;
          const int64_t at = (int64_t)m * ldc + n;
          f32x4 v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
          if (vector && n + 4 <= n_valid) {
            if (mul) v *= *reinterpret_cast<const f32x4*>(mul + at);
            *reinterpret_cast<f32x4*>(out + at) = v;
          } else {
#pragma unroll
            for (int q = 0; q < 4; q++)
              if (n + q < n_valid) out[at + q] = mul ? v[q] * mul[at + q] : v[q];
          }
        }
      }
  }
};

struct SddArgs {
  const float* lhs;
  int64_t lsm, lsk;
  const float* rhs;
  int64_t rsk, rsn;
  int k;
  float* out;
  const void* row_indices;
  const void* column_indices;
  int idx32;
  int activation;
  const float* multiplier;
};

template <int BLK>
__global__ __launch_bounds__(kThreads) void sdd_kernel(SddArgs g) {
  __shared__ float lds[Tile<BLK>::kLdsFloats];
  const int64_t p = blockIdx.x;
  const int64_t r = load_index(g.row_indices, p, g.idx32), c = load_index(g.column_indices, p, g.idx32);
  Tile<BLK> t;
  t.clear();
  t.accumulate(g.lhs + r * BLK * g.lsm, g.lsm, g.lsk, BLK, g.rhs + c * BLK * g.rsn, g.rsk, g.rsn, BLK, g.k, lds);
  t.store(g.out + p * BLK * BLK, BLK, BLK, BLK, g.activation, g.multiplier ? g.multiplier + p * BLK * BLK : nullptr);
}

// One line of op(S) against a BLK-wide tile of the dense operand.  SPARSE_LHS: dsd (the line is a block row of op(S),
// the dense operand is the rhs); otherwise dds (the line is a block column, the dense operand is the lhs).
struct WalkArgs {
  const float* data;
  const int32_t* walk_offsets;
  const void* walk_positions;
  const int32_t* walk_blocks;  // indirect block ids, or null: the entry number is the block id
  const float* dense;
  int64_t ds_outer, ds_k;      // dense element strides: along its free dimension (n of the rhs, m of the lhs) and along k
  int64_t bs_mn, bs_k;         // element strides inside a stored block: along the line's own dimension and along k
  float* out;
  int64_t ldc;
  int free_extent;             // n (dsd) or m (dds)
  int idx32;
};

template <int BLK, bool SPARSE_LHS>
__global__ __launch_bounds__(kThreads) void walk_kernel(WalkArgs g) {
  __shared__ float lds[Tile<BLK>::kLdsFloats];
  const int tiles = (g.free_extent + BLK - 1) / BLK;
  const int line = blockIdx.x / tiles, f0 = (blockIdx.x % tiles) * BLK;
  const int valid = g.free_extent - f0 < BLK ? g.free_extent - f0 : BLK;
  Tile<BLK> t;
  t.clear();
  const int begin = g.walk_offsets[line], end = g.walk_offsets[line + 1];
  for (int e = begin; e < end; e++) {
    const int64_t kb = load_index(g.walk_positions, e, g.idx32);
    const float* blk = g.data + (int64_t)(g.walk_blocks ? g.walk_blocks[e] : e) * BLK * BLK;
    const float* dense = g.dense + kb * BLK * g.ds_k + (int64_t)f0 * g.ds_outer;
    if constexpr (SPARSE_LHS) t.accumulate(blk, g.bs_mn, g.bs_k, BLK, dense, g.ds_k, g.ds_outer, valid, BLK, lds);
    else t.accumulate(dense, g.ds_outer, g.ds_k, valid, blk, g.bs_k, g.bs_mn, BLK, BLK, lds);
  }
  if constexpr (SPARSE_LHS) t.store(g.out + (int64_t)line * BLK * g.ldc + f0, g.ldc, BLK, valid, kNoActivation, nullptr);
  else t.store(g.out + (int64_t)f0 * g.ldc + (int64_t)line * BLK, g.ldc, valid, BLK, kNoActivation, nullptr);
}

// ---------------------------------------------------------------------------
// Fast set.
//
// An operand tile is EXT (m or n extent) x kFastKT k, in LDS as it lies in memory: K-major [EXT][32 k], 128-byte rows,
// or MN-major [32 k][EXT].  A wavefront's 1 KiB transfer fills consecutive LDS bytes, so the swizzles that keep the
// reads free of bank conflicts are applied by choosing which 16-byte piece a lane fetches.  In a group of eight k the
// lanes of the lower half hold k 0..3 and those of the upper half k 4..7: a K-major operand is then read as one
// 16-byte piece per lane for four MFMAs, an MN-major one as a 4-byte word per MFMA.
// ---------------------------------------------------------------------------
constexpr int kFastKT = 32;

template <int EXT, bool KMAJOR>
struct FastOperand {
  static constexpr int kBytes = EXT * kFastKT * 4;
  static constexpr int kSlices = kBytes / 1024;
  static constexpr int kPerWave = kSlices / 4;
  static_assert(kSlices % 4 == 0, "whole transfers per wavefront");
  // Byte offset from the tile's origin of what lane `lane` fetches for slice `slice`; ld in elements.
  __device__ __forceinline__ static uint32_t source(int slice, int lane, int64_t ld) {
    if constexpr (KMAJOR) {
      const int row = slice * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
      return (uint32_t)((row * ld + piece * 4) * 4);
    } else {
      constexpr int kPieces = EXT / 4;  // per k row
      const int k = slice * (64 / kPieces) + lane / kPieces;
      const int byte = ((lane % kPieces) << 4) ^ swizzle(k);
      return (uint32_t)(k * ld * 4 + byte);
    }
  }
  // Rows k and k + 4 are read together, 128 bytes of each: when the rows are multiples of the 256 bytes of banks apart
  // the second one is kept with its 128-byte halves swapped.
  __device__ __forceinline__ static int swizzle(int k) { return EXT >= 64 ? ((k >> 2) & 1) << 7 : 0; }
  // f[j] = element (mn + lane % 32, k = 8 group + 4 (lane / 32) + j)
  __device__ __forceinline__ static void frag(const char* s, int mn, int group, int lane, float (&f)[4]) {
    if constexpr (KMAJOR) {
      const int row = mn + (lane & 31), piece = (2 * group + (lane >> 5)) ^ ((row >> 1) & 7);
      const f32x4 v = *reinterpret_cast<const f32x4*>(s + row * 128 + piece * 16);
#pragma unroll
      for (int j = 0; j < 4; j++) f[j] = v[j];
    } else {
      const int k = 8 * group + 4 * (lane >> 5);
      const char* at = s + k * (EXT * 4) + ((4 * (mn + (lane & 31))) ^ swizzle(k));
#pragma unroll
      for (int j = 0; j < 4; j++) f[j] = *reinterpret_cast<const float*>(at + j * (EXT * 4));
    }
  }
};

// T x T output tile of four wavefronts: 2 x 2 of (T / 2) x (T / 2), or for T = 32 one tile whose K-tiles are split over
// the wavefronts (8 k each) and added up at the end, in the order of the wavefronts.
template <int T, bool AK, bool BK>
struct Fast {
  static constexpr int kStages = T == 128 ? 2 : T == 64 ? 3 : 4;
  static constexpr int kW = T == 128 ? 2 : 1;  // 32x32 MFMA tiles per wavefront in each direction
  static constexpr bool kSplit = T == 32;
  using OpA = FastOperand<T, AK>;
  using OpB = FastOperand<T, BK>;
  static constexpr int kStageBytes = OpA::kBytes + OpB::kBytes;
  static constexpr int kLds = kStages * kStageBytes;  // (T = 32: 32 KiB, of which the partial sums use 16)
  static constexpr int kLoads = OpA::kPerWave + OpB::kPerWave;
  f32x16_t acc[kW][kW];

  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < kW; i++)
#pragma unroll
      for (int j = 0; j < kW; j++) acc[i][j] = f32x16_t{};
  }

  // acc += the `ntiles` K-tiles whose origins tile_fn(t, a, b) gives (called once per t, in increasing order)
  template <class TileFn>
  __device__ __forceinline__ void accumulate(int ntiles, int64_t lda, int64_t ldb, char* smem, TileFn&& tile_fn) {
    const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
    const uint32_t lds0 = (uint32_t)(uintptr_t)((STK_LDS char*)smem);
    uint32_t offa[OpA::kPerWave], offb[OpB::kPerWave];
#pragma unroll
    for (int i = 0; i < OpA::kPerWave; i++) offa[i] = OpA::source(i * 4 + wave, lane, lda);
#pragma unroll
    for (int i = 0; i < OpB::kPerWave; i++) offb[i] = OpB::source(i * 4 + wave, lane, ldb);
    auto issue = [&](int t) {
      const float *a, *b;
      tile_fn(t, a, b);
      const gptr_t ga = uniform_global(a), gb = uniform_global(b);
      const uint32_t stage = lds0 + (uint32_t)(t % kStages) * kStageBytes;
#pragma unroll
      for (int i = 0; i < OpA::kPerWave; i++) dma16(ga, offa[i], stage + (i * 4 + wave) * 1024);
#pragma unroll
      for (int i = 0; i < OpB::kPerWave; i++) dma16(gb, offb[i], stage + OpA::kBytes + (i * 4 + wave) * 1024);
    };
#pragma unroll
    for (int t = 0; t < kStages - 1; t++)
      if (t < ntiles) issue(t);
    const int m0 = kSplit ? 0 : (wave & 1) * (T / 2), n0 = kSplit ? 0 : (wave >> 1) * (T / 2);
    for (int t = 0; t < ntiles; t++) {
      // K-tile t has landed; up to kStages - 2 younger ones may stay in flight
      const int younger = ntiles - 1 - t;
      if (kStages >= 4 && younger >= 2) wait_vmcnt<2 * kLoads>();
      else if (kStages >= 3 && younger >= 1) wait_vmcnt<1 * kLoads>();
      else wait_vmcnt<0>();
      __syncthreads();  // every wavefront's part of K-tile t is there, and K-tile t - 1, whose stage is refilled, has been read
      if (t + kStages - 1 < ntiles) issue(t + kStages - 1);
      const char* sa = smem + (t % kStages) * kStageBytes;
      const char* sb = sa + OpA::kBytes;
#pragma unroll
      for (int g = 0; g < (kSplit ? 1 : 4); g++) {
        const int group = kSplit ? wave : g;
        float fa[kW][4], fb[kW][4];
#pragma unroll
        for (int i = 0; i < kW; i++) OpA::frag(sa, m0 + 32 * i, group, lane, fa[i]);
#pragma unroll
        for (int j = 0; j < kW; j++) OpB::frag(sb, n0 + 32 * j, group, lane, fb[j]);
        // operands swapped, as in the 16-bit engine: a lane then owns four consecutive columns of one output row
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
          for (int i = 0; i < kW; i++)
#pragma unroll
            for (int j = 0; j < kW; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j][q], fa[i][q], acc[i][j], 0, 0, 0);
      }
    }
    __syncthreads();  // the ring has been read: it is filled again, or used for the partial sums
  }

  // out[m * ldc + n] = act(acc) (* mul[m * ldc + n]); out and mul 16-byte aligned with rows at multiples of 16 bytes
  __device__ __forceinline__ void store(float* out, int64_t ldc, int activation, const float* mul, char* smem) {
    const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
    auto put = [&](int m, int n, f32x4 v) {
      const int64_t at = (int64_t)m * ldc + n;
      if (mul) v *= *reinterpret_cast<const f32x4*>(mul + at);
      *reinterpret_cast<f32x4*>(out + at) = v;
    };
    if constexpr (kSplit) {
      // wavefront w finishes the columns 8 w + 0..7: values 4 w .. 4 w + 3 of every lane
      float* part = reinterpret_cast<float*>(smem);
#pragma unroll
      for (int r = 0; r < 16; r++) part[(wave * 16 + r) * 64 + lane] = acc[0][0][r];
      __syncthreads();
      f32x16_t v = {};
#pragma unroll
      for (int q = 0; q < 4; q++) {
        float sum = part[(4 * wave + q) * 64 + lane];
#pragma unroll
        for (int w = 1; w < 4; w++) sum += part[(w * 16 + 4 * wave + q) * 64 + lane];
        v[q] = sum;
      }
      if (activation != kNoActivation) activate_all(v, activation);
      put(lane & 31, 8 * wave + 4 * (lane >> 5), f32x4{v[0], v[1], v[2], v[3]});
    } else {
      const int m0 = (wave & 1) * (T / 2), n0 = (wave >> 1) * (T / 2);
#pragma unroll
      for (int i = 0; i < kW; i++)
#pragma unroll
        for (int j = 0; j < kW; j++) {
          if (activation != kNoActivation) activate_all(acc[i][j], activation);
#pragma unroll
          for (int g = 0; g < 4; g++)
            put(m0 + 32 * i + (lane & 31), n0 + 32 * j + 8 * g + 4 * (lane >> 5),
                f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]});
        }
    }
  }
};

template <int BLK, int T, bool AK, bool BK>
__global__ __launch_bounds__(kThreads, 2) void sdd_fast_kernel(SddArgs g, int nnz) {
  __shared__ __align__(16) char smem[Fast<T, AK, BK>::kLds];
  constexpr int kSide = BLK / T, kPerBlock = kSide * kSide;
  const int item = xcd_chunked(blockIdx.x, nnz * kPerBlock);
  const int p = item / kPerBlock, m0 = item % kPerBlock / kSide * T, n0 = item % kSide * T;
  const int64_t r = uniform(load_index(g.row_indices, p, g.idx32)), c = uniform(load_index(g.column_indices, p, g.idx32));
  const float* a0 = g.lhs + (r * BLK + m0) * g.lsm;
  const float* b0 = g.rhs + (c * BLK + n0) * g.rsn;
  Fast<T, AK, BK> t;
  t.clear();
  t.accumulate(g.k / kFastKT, AK ? g.lsm : g.lsk, BK ? g.rsn : g.rsk, smem, [&](int i, const float*& a, const float*& b) {
    a = a0 + (int64_t)i * kFastKT * g.lsk;
    b = b0 + (int64_t)i * kFastKT * g.rsk;
  });
  const int64_t at = (int64_t)p * BLK * BLK + m0 * BLK + n0;
  t.store(g.out + at, BLK, g.activation, g.multiplier ? g.multiplier + at : nullptr, smem);
}

// Which tile workgroup `block` computes: line, stretch of the line, tile of the dense operand.  A line takes as long as it
// has blocks, and a launch with one tile per compute unit as long as its longest line, so the lines are spread evenly over
// the dies - every die takes all lines for its eighth of the dense operand - and a die's workgroups come longest line first,
// every second round of its compute units in reverse, so that the units, which hold several small tiles at once, get about
// equal sums.  More than 64 lines are left in their order: there are enough tiles for the dispatch to even them out.
struct WalkItem {
  int line, stretch, tile;
};
template <int SIDE>
__device__ __forceinline__ WalkItem walk_item(const int32_t* offsets, int lines, int tiles, int items) {
  constexpr int kDies = 8, kUnitsPerDie = 32;
  const int lane = threadIdx.x & 63, block = uniform((int)blockIdx.x);
  if (lines > 64) {
    const int item = xcd_chunked(block, items);
    return {item / (SIDE * tiles), item % SIDE, item / SIDE % tiles};
  }
  const int die = block % kDies, on_die = (items - die + kDies - 1) / kDies;
  int at = block / kDies;
  if ((at / kUnitsPerDie) % 2 == 1 && (at / kUnitsPerDie + 1) * kUnitsPerDie <= on_die)
    at = at / kUnitsPerDie * kUnitsPerDie + kUnitsPerDie - 1 - at % kUnitsPerDie;
  int rank, rest;   // rank of the line by length; stretch and tile
  if (tiles % kDies == 0) {
    const int per_line = SIDE * (tiles / kDies);
    rank = at / per_line, rest = at % per_line + die * per_line;
  } else {
    const int item = at * kDies + die;
    rank = item / (SIDE * tiles), rest = item % (SIDE * tiles);
  }
  // lane i: the length of line i and how many lines come before it
  const int mine = lane < lines ? offsets[lane + 1] - offsets[lane] : -1;
  int before = 0;
  for (int i = 0; i < lines; i++) {
    const int other = __builtin_amdgcn_readlane(mine, i);
    before += other > mine || (other == mine && i < lane);
  }
  const int line = (int)__ffsll((unsigned long long)__ballot(lane < lines && before == rank)) - 1;
  return {line, rest % SIDE, rest / SIDE};
}

// One T-wide stretch of a line of op(S) against a T-wide tile of the dense operand.
template <int BLK, int T, bool SPARSE_LHS, bool AK, bool BK>
__global__ __launch_bounds__(kThreads, 2) void walk_fast_kernel(WalkArgs g, int lines, int items) {
  __shared__ __align__(16) char smem[Fast<T, AK, BK>::kLds];
  constexpr int kSide = BLK / T, kPer = BLK / kFastKT;
  const WalkItem item = walk_item<kSide>(g.walk_offsets, lines, g.free_extent / T, items);
  const int line = uniform(item.line), f0 = uniform(item.tile) * T, l0 = uniform(item.stretch) * T;
  const int lane = threadIdx.x & 63;
  const int begin = uniform(g.walk_offsets[line]), end = uniform(g.walk_offsets[line + 1]);
  const float* dense0 = g.dense + (int64_t)f0 * g.ds_outer;
  const float* data0 = g.data + (int64_t)l0 * g.bs_mn;
  Fast<T, AK, BK> t;
  t.clear();
  for (int s0 = begin; s0 < end; s0 += 64) {
    const int count = end - s0 < 64 ? end - s0 : 64;
    // lane i holds the place and the block of walk entry s0 + i: the K loop gets them with a lane read
    const int e = s0 + (lane < count ? lane : count - 1);
    const int seg_k = load_index(g.walk_positions, e, g.idx32), seg_block = g.walk_blocks ? g.walk_blocks[e] : e;
    auto origins = [&](int i, const float*& a, const float*& b) {
      const int sub = i % kPer * kFastKT;
      const float* block = data0 + (int64_t)__builtin_amdgcn_readlane(seg_block, i / kPer) * BLK * BLK + sub * g.bs_k;
      const float* dense = dense0 + ((int64_t)__builtin_amdgcn_readlane(seg_k, i / kPer) * BLK + sub) * g.ds_k;
      a = SPARSE_LHS ? block : dense;
      b = SPARSE_LHS ? dense : block;
    };
    const int64_t ld_block = BLK, ld_dense = g.ds_k == 1 ? g.ds_outer : g.ds_k;
    t.accumulate(count * kPer, SPARSE_LHS ? ld_block : ld_dense, SPARSE_LHS ? ld_dense : ld_block, smem, origins);
  }
  const int64_t row = SPARSE_LHS ? (int64_t)line * BLK + l0 : f0, col = SPARSE_LHS ? f0 : (int64_t)line * BLK + l0;
  t.store(g.out + row * g.ldc + col, g.ldc, kNoActivation, nullptr, smem);
}

// Side of the output tiles for a problem of `area` tiles of 32 x 32 whose extents are multiples of `most`.  The matrix pipe
// is the bound, so a tile that leaves compute units without work, or with a longer line than others have, costs in
// proportion, while a smaller tile than needed moves more operand bytes per FLOP.  Kernel times in us with tiles of 128 /
// 64 / 32:
//   sdd, 32 blocks of 128, k = 1024 (32 / 128 / 512 tiles)            66 / 24 / 15
//   sdd, 64 blocks of 128, k = 2048 (64 / 256 / 1024 tiles)            - / 49 / 45
//   dsd, 1024 x 1024 half full x 1024 (64 / 256 / 1024 tiles)         69 / 27 / 17
//   dsd, 1536 x 640, 30 % full, x 896 (84 / 336 / 1344 tiles)          - / 14 / 12
//   sdd, 128 blocks of 128, k = 2048 (128 / 512 / 2048 tiles)          - / 77 / 85
//   dsd, 2048 x 2048, a quarter full, x 2048 (256 / 1024 / 4096 tiles) - / 52 / 58
//   dds, 3072 x 3072 half full, 2048 rows (384 / 1536 / 6144 tiles)  254 / 165 / 207
//   dsd, 4096 x 4096 half full x 4096 (1024 / 4096 / 16384 tiles)    521 / 566 / 719
// so 64 as soon as every unit gets two tiles, 128 from four of them for every unit on.  (Before these kernels, with a
// 128 x 128 tile per block in all of these cases: sdd 69, dsd 68, and 990 for the dsd of 4096 x 4096; with the lines in their
// order, a line on one die, the dsd of 1024 x 1024 took 26 us with tiles of 64 and 27 with tiles of 32.)
inline int fast_tile(int64_t area, int most) {
  const int64_t units = compute_units() > 0 ? compute_units() : 256;
  if (most >= 128 && area / 16 >= 4 * units) return 128;
  return most >= 64 && area / 4 >= 2 * units ? 64 : 32;
}

// A float32 array that the transfers can read: unit stride in one dimension, the other one and the base multiples of 16
// bytes, and rows of a tile within 32-bit byte offsets of its origin.
inline bool fast_layout(const void* p, int64_t s0, int64_t s1) {
  const int64_t ld = s1 == 1 ? s0 : s1;
  return aligned16(p) && (s0 == 1 || s1 == 1) && ld > 0 && ld % 4 == 0 && ld < (1 << 22);
}

}  // namespace f32

int sdd_f32(const void* lhs, int64_t lhs_stride_m, int64_t lhs_stride_k, const void* rhs, int64_t rhs_stride_k, int64_t rhs_stride_n,
            int64_t m, int64_t k, int64_t n, void* out, const void* row_indices, const void* column_indices, int64_t nnz,
            int blocking, int index_dtype, int activation, const void* multiplier, hipStream_t stream) {
  if (activation < 0 || activation >= kActivations) return fail(STK_ERR_UNSUPPORTED, "stk_sdd: activation %d", activation);
  if (blocking != 64 && blocking != 128) return fail(STK_ERR_UNSUPPORTED, "stk_sdd: blocking %d (64 or 128)", blocking);
  if (index_dtype != STK_I16 && index_dtype != STK_I32) return fail(STK_ERR_UNSUPPORTED, "stk_sdd: index dtype %d", index_dtype);
  if (m < 0 || n < 0 || k < 0 || nnz < 0) return fail(STK_ERR_DIMS, "stk_sdd: negative size");
  if (m % blocking || n % blocking || k % 32)
    return fail(STK_ERR_DIMS, "incompatible dimensions: [%lld, %lld] x [%lld, %lld] with blocking %d (m, n must be divisible by the blocking, k by 32)",
                (long long)m, (long long)k, (long long)k, (long long)n, blocking);
  if (k > INT32_MAX || nnz > INT32_MAX) return fail(STK_ERR_UNSUPPORTED, "stk_sdd: size exceeds 32-bit range");
  if (nnz == 0) return STK_OK;
  if (!lhs || !rhs || !out || !row_indices || !column_indices) return fail(STK_ERR_DIMS, "stk_sdd: missing pointer");
  const f32::SddArgs g{static_cast<const float*>(lhs), lhs_stride_m, lhs_stride_k, static_cast<const float*>(rhs), rhs_stride_k, rhs_stride_n,
                       (int)k, static_cast<float*>(out), row_indices, column_indices, index_dtype == STK_I32, activation,
                       static_cast<const float*>(multiplier)};
  if (f32::fast_layout(lhs, lhs_stride_m, lhs_stride_k) && f32::fast_layout(rhs, rhs_stride_k, rhs_stride_n) && aligned16(out) && (!multiplier || aligned16(multiplier))) {
    const int t = f32::fast_tile(nnz * (blocking / 32) * (blocking / 32), blocking);
    const bool ak = lhs_stride_k == 1, bk = rhs_stride_n != 1;
    const int64_t grid = nnz * (blocking / t) * (blocking / t);
    if (grid <= INT32_MAX) {
#define STK_F32_SDD(BLK, T, AK, BK)                                                                                              \
  if (blocking == BLK && t == T && ak == AK && bk == BK)                                                                         \
    hipLaunchKernelGGL((f32::sdd_fast_kernel<BLK, T, AK, BK>), dim3((unsigned)grid), dim3(f32::kThreads), 0, stream, g, (int)nnz);
#define STK_F32_SDD_LAYOUTS(BLK, T) STK_F32_SDD(BLK, T, true, true) STK_F32_SDD(BLK, T, true, false) STK_F32_SDD(BLK, T, false, true) STK_F32_SDD(BLK, T, false, false)
      STK_F32_SDD_LAYOUTS(128, 128) STK_F32_SDD_LAYOUTS(128, 64) STK_F32_SDD_LAYOUTS(128, 32) STK_F32_SDD_LAYOUTS(64, 64) STK_F32_SDD_LAYOUTS(64, 32)
#undef STK_F32_SDD_LAYOUTS
#undef STK_F32_SDD
      return check_launch("stk_sdd");
    }
  }
  if (blocking == 128) hipLaunchKernelGGL(f32::sdd_kernel<128>, dim3((unsigned)nnz), dim3(f32::kThreads), 0, stream, g);
  else hipLaunchKernelGGL(f32::sdd_kernel<64>, dim3((unsigned)nnz), dim3(f32::kThreads), 0, stream, g);
  return check_launch("stk_sdd");
}

// dsd (sparse_lhs) or dds on float32 values over the `lines` walked lines of op(S); `free_extent` is n of the rhs (dsd)
// or m of the lhs (dds), with element strides (dense_stride_free, dense_stride_k).  line_major: the rows of a stored
// block run along the walked line's own dimension (dsd of S, dds of S^T); otherwise along k (dsd of S^T, dds of S).
int walk_f32(bool sparse_lhs, const char* who, int64_t lines, int64_t free_extent, const void* data, const int32_t* walk_offsets,
             const void* walk_positions, const int32_t* walk_blocks, bool line_major, const void* dense, int64_t dense_stride_free,
             int64_t dense_stride_k, void* out, int64_t out_stride_m, int64_t nnz, int blocking, int index_dtype, hipStream_t stream) {
  if (blocking != 64 && blocking != 128) return fail(STK_ERR_UNSUPPORTED, "%s: blocking %d (64 or 128)", who, blocking);
  if (index_dtype != STK_I16 && index_dtype != STK_I32) return fail(STK_ERR_UNSUPPORTED, "%s: index dtype %d", who, index_dtype);
  if (lines == 0 || free_extent == 0) return STK_OK;
  const int64_t tiles = (free_extent + blocking - 1) / blocking;
  if (lines * tiles > INT32_MAX || free_extent > INT32_MAX) return fail(STK_ERR_UNSUPPORTED, "%s: size exceeds 32-bit range", who);
  if (!walk_offsets || !out || (nnz > 0 && (!walk_positions || !data || !dense))) return fail(STK_ERR_DIMS, "%s: missing metadata pointer", who);
  const int64_t b = blocking;
  const f32::WalkArgs g{static_cast<const float*>(data), walk_offsets, walk_positions, walk_blocks, static_cast<const float*>(dense),
                        dense_stride_free, dense_stride_k, line_major ? b : 1, line_major ? 1 : b,
                        static_cast<float*>(out), out_stride_m, (int)free_extent, index_dtype == STK_I32};
  const int side = free_extent % 128 == 0 ? 128 : free_extent % 64 == 0 ? 64 : free_extent % 32 == 0 ? 32 : 0;
  if (side && f32::fast_layout(dense, dense_stride_free, dense_stride_k) && aligned16(data) && aligned16(out) && out_stride_m % 4 == 0) {
    const int t = f32::fast_tile(lines * (b / 32) * (free_extent / 32), side < blocking ? side : blocking);
    const int64_t items = lines * (b / t) * (free_extent / t);
    if (items <= INT32_MAX) {
      // K-major operands: stored blocks whose rows run along the line, a dense operand with unit stride along k
      const bool sk = line_major, dk = dense_stride_k == 1;
#define STK_F32_WALK(BLK, T, SL, SK, DK)                                                                                               \
  if (blocking == BLK && t == T && sparse_lhs == SL && sk == SK && dk == DK)                                                           \
    hipLaunchKernelGGL((f32::walk_fast_kernel<BLK, T, SL, SL ? SK : DK, SL ? DK : SK>), dim3((unsigned)items), dim3(f32::kThreads), 0, stream, g, (int)lines, (int)items);
#define STK_F32_WALK_LAYOUTS(BLK, T, SL) STK_F32_WALK(BLK, T, SL, true, true) STK_F32_WALK(BLK, T, SL, true, false) STK_F32_WALK(BLK, T, SL, false, true) STK_F32_WALK(BLK, T, SL, false, false)
#define STK_F32_WALKS(BLK, T) STK_F32_WALK_LAYOUTS(BLK, T, true) STK_F32_WALK_LAYOUTS(BLK, T, false)
      STK_F32_WALKS(128, 128) STK_F32_WALKS(128, 64) STK_F32_WALKS(128, 32) STK_F32_WALKS(64, 64) STK_F32_WALKS(64, 32)
#undef STK_F32_WALKS
#undef STK_F32_WALK_LAYOUTS
#undef STK_F32_WALK
      return check_launch(who);
    }
  }
  const dim3 grid((unsigned)(lines * tiles));
  if (sparse_lhs) {
    if (blocking == 128) hipLaunchKernelGGL((f32::walk_kernel<128, true>), grid, dim3(f32::kThreads), 0, stream, g);
    else hipLaunchKernelGGL((f32::walk_kernel<64, true>), grid, dim3(f32::kThreads), 0, stream, g);
  } else {
    if (blocking == 128) hipLaunchKernelGGL((f32::walk_kernel<128, false>), grid, dim3(f32::kThreads), 0, stream, g);
    else hipLaunchKernelGGL((f32::walk_kernel<64, false>), grid, dim3(f32::kThreads), 0, stream, g);
  }
  return check_launch(who);
}

}  // namespace stk
