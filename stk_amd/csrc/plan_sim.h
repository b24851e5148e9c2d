// The choice of slices for the last round of a stk_dsd launch, shared by the two builders of fusion plans (plan.hip,
// dmoe.hip): a simulation of the hardware's dispatch.
#pragma once
#include "common.h"

namespace stk {

// When the tiles of a launch fill the compute units a few times only, the last round
// leaves most of them idle.  Cutting the tiles of that round into k slices along the
// contraction (workgroups add the partial tiles up) fills the round better, at the price of
// the partial tiles' round trip through memory.  Which k pays is found by playing the
// hardware's dispatch through: workgroups start in order, each on the compute unit that
// is free first.  Tiles of one kind take equally long here (the lines' average length), so
// the compute units are kept as a few groups (free time, how many) in ascending order.
constexpr int kSimGroups = 24;    // groups alive at a time
constexpr int kSimCapacity = 48;  // room for the queue to move along before it is shifted back
struct HostSim {
  float time[kSimCapacity];
  int count[kSimCapacity];
  int head, tail;  // the groups are entries [head, tail), ascending in time
  void reset(int units) { time[0] = 0.f, count[0] = units, head = 0, tail = 1; }
  // n work items of the same duration
  void run(int n, float duration) {
    while (n > 0) {
      const int m = n < count[head] ? n : count[head];
      const float t = time[head] + duration;
      n -= m;
      count[head] -= m;
      if (count[head] == 0) head++;
      if (tail == kSimCapacity) {
        for (int i = head; i < tail; i++) time[i - head] = time[i], count[i - head] = count[i];
        tail -= head, head = 0;
      }
      int at = tail;
      while (at > head && time[at - 1] > t) at--;
      if (at > head && time[at - 1] == t) {
        count[at - 1] += m;
      } else if (tail - head == kSimGroups) {
        // out of groups: join a neighbour (a small error in a rare case)
        count[at < tail ? at : tail - 1] += m;
      } else {
        for (int i = tail; i > at; i--) time[i] = time[i - 1], count[i] = count[i - 1];
        time[at] = t, count[at] = m, tail++;
      }
    }
  }
  float end() const { return time[tail - 1]; }
};

// The same by a wavefront: lane i holds group i, in ascending order of time.  A step is a few lane reads, a ballot and at
// most two moves of all groups by one lane, some 150 cycles; with the groups in LDS, one simulation per thread, it was a
// chain of LDS accesses of some 1500 cycles, which made the simulation most of the time of a plan.
struct WaveSim {
  float time;
  int count, groups;  // groups: how many lanes hold one
  __device__ __forceinline__ void reset(int units) {
    time = 0.f, count = units, groups = 1;
  }
  __device__ __forceinline__ void run(int n, float duration) {
    const int lane = threadIdx.x & 63;
    while (n > 0) {
      const int first = __builtin_amdgcn_readlane(count, 0);
      const float t = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, time), 0)) + duration;
      const int m = n < first ? n : first;
      n -= m;
      if (m == first) {
        time = __shfl_down(time, 1, 64), count = __shfl_down(count, 1, 64);
        groups--;
      } else if (lane == 0) {
        count -= m;
      }
      const int at = __popcll(__ballot(lane < groups && time <= t));
      const bool joins = at > 0 && __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, time), at > 0 ? at - 1 : 0)) == t;
      if (joins || groups == kSimGroups) {
        const int to = joins ? at - 1 : (at < groups ? at : groups - 1);
        if (lane == to) count += m;
      } else {
        const float above_time = __shfl_up(time, 1, 64);
        const int above_count = __shfl_up(count, 1, 64);
        if (lane > at) time = above_time, count = above_count;
        if (lane == at) time = t, count = m;
        groups++;
      }
    }
  }
  __device__ __forceinline__ float end() const { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, time), groups - 1)); }
};

// Simulated end of a launch whose last round is cut into k slices.  tiles[]: pairs, threes, lone lines;
// length: average blocks per line.
template <class Sim>
__host__ __device__ inline float simulate_launch(Sim& sim, const int (&tiles)[3], float length, int units, int k) {
  // Durations in units of one block of k of a 256x256 tile (about 5 us).  Measured on an MI355X: a workgroup
  // spends about 4 such units outside its K loop (start, first loads, store), and 2 more when its tile is a
  // slice (partial tile out to memory and back in, the counter); 384x128 and 128x256 tiles take 0.75 and 0.58
  // of a 256x256 tile's time per block.
  const float start = 4.f, seam = 2.f;
  const float duration[3] = {length, 0.75f * length, 0.58f * length};
  const int total = tiles[0] + tiles[1] + tiles[2];
  const int whole = (total - 1) / units * units;
  sim.reset(units);
  int left = whole, tail[3];
  for (int kind = 0; kind < 3; kind++) {
    const int n = tiles[kind] < left ? tiles[kind] : left;
    sim.run(n, duration[kind] + start);
    left -= n;
    tail[kind] = tiles[kind] - n;
  }
  for (int slice = 0; slice < k; slice++)
    for (int kind = 0; kind < 3; kind++) sim.run(tail[kind], k == 1 ? duration[kind] + start : duration[kind] / k + start + seam);
  return sim.end();
}

// With more than four rounds of tiles the last one matters too little to be worth the simulation.
__host__ __device__ inline bool tail_slices_considered(int64_t tiles, int units) { return tiles > 0 && units > 0 && tiles <= 4 * (int64_t)units; }

// Slices for the tiles of the last round, given the simulated ends for k = 1 .. kMaxTailSlices: the k with the
// shortest launch, 1 unless k > 1 saves 2 %.
__host__ __device__ inline int choose_tail_slices(const float (&end)[kMaxTailSlices]) {
  int best = 1;
  float best_end = end[0];
  for (int k = 2; k <= kMaxTailSlices; k++)
    if (end[k - 1] < best_end && end[k - 1] < 0.98f * end[0]) best = k, best_end = end[k - 1];
  return best;
}

}  // namespace stk
