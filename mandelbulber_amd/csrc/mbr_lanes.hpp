// mbr_lanes.hpp — how the persistent kernels share out their work: the queues
// that hand items to the lanes of a wave, the loop that keeps lanes busy with
// distance estimates of different lengths, and the launch of such a kernel.
#pragma once

#include <algorithm>
#include <atomic>

#include "mbr_kernels.hpp"

namespace mbr {

constexpr int kBlock = 256;

// A lane wants an item, runs an estimate, has an estimate complete, or found
// the queue empty.
enum : int { MS_NEED = 0, MS_ITER = 1, MS_DONE = 2, MS_EXHAUSTED = 3 };

// Cancel polling (mbr_cancel, the reference's programClosed test per pixel,
// src/Render3D.cpp:369-378).  A band's work queue carries the stop in its
// counter: kStopBit, set by whoever read the host flag (poll_cancel, a read
// over the bus, so not for every hand-out) and found it set.
//   k_band_reset  reads the flag before the march, the surface kernel before
//                 AO: a wave that builds its queue sees a stop from before
//                 its kernel, so also its fixed first items are dropped
//   hand-outs     from the shared counter return the bit with their add; those
//                 that cross a multiple of 2^poll_shift read the flag
// (Hand-outs from a run taken before do not load the counter: with a load for
// every hit a 1080p frame with AO took 13.0 ms instead of 9.3, loads and adds to
// one address being served one after the other.  Polled queues take shorter
// runs instead.)
constexpr unsigned long long kStopBit = 1ull << 48;

// By one lane: whether the flag is set; the queue then carries the stop.
__device__ __forceinline__ bool poll_cancel(const BandBufs &b, unsigned long long *queue) {
  if (!b.cancel || *b.cancel == 0) return false;
  atomicOr(queue, kStopBit);
  return true;
}

__device__ __forceinline__ bool crosses(long long first, long long n, int poll_shift) {
  return ((first + n) >> poll_shift) != (first >> poll_shift);
}

// Lane 0's value, in scalar registers (what the queue keeps is the wave's).
__device__ __forceinline__ unsigned long long first_lane(unsigned long long v) {
  return (unsigned)__builtin_amdgcn_readfirstlane((int)v) |
         (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32;
}

// Lanes of a wave that take items, for n items over the launch's waves: few
// items spread over half of the waves, at least 4 each, so that a wave's
// passes wait for fewer lanes.
__device__ __forceinline__ int item_lanes(long long n) {
  const long long half = (long long)gridDim.x * (kBlock / 128);
  const long long per = (n + half - 1) / half;
  return per >= 64 ? 64 : per < 4 ? 4 : (int)per;
}

// A wave's share of the band's n items (rays, hits): its first `lanes` items by
// its number, then runs taken from a counter shared by all waves.  Adds to one
// address pass at about 13 ns each on MI355X, whichever wave sends them: with
// an add for every hand-out, 8192 waves spent 100 us just to find a small
// frame's queue empty, so an item costs no add where there are lanes for all,
// and a run grows with what is left (up to max_run, and so that every wave of
// the launch can still take 4 runs).
// Poll: hand-outs poll the cancel flag every 2^poll_shift items of the counter.
template <bool Poll = false>
struct WaveQueue {
  unsigned long long *queue;
  long long n, cur, end, shared;  // shared: first item handed out by the counter
  int waves, max_run, poll_shift;
  bool dry, stopped;  // stopped (Poll): the band was

  __device__ __forceinline__ WaveQueue(unsigned long long *queue_, long long n_, int lanes, int max_run_ = 256,
                                       int poll_shift_ = 0) {
    queue = queue_;
    n = n_;
    max_run = max_run_;
    poll_shift = poll_shift_;
    // what the kernels before left there, as a scalar load (first_lane keeps the
    // compiler from a narrower vector load, which queues behind the adds of the
    // waves that started first: 100 us of a 2.1 ms frame)
    stopped = Poll && (first_lane(*queue) & kStopBit);
    waves = (int)gridDim.x * (kBlock / 64);
    // workgroups first, so that few items spread over the CUs
    const long long w = (long long)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * gridDim.x + blockIdx.x;
    cur = w * lanes;
    end = cur + lanes;
    shared = (long long)waves * lanes;
    if (cur > n) cur = n;
    if (end > n) end = n;
    dry = shared >= n;
  }
  // For the whole wave: lane `rank` of `need` lanes gets its item, or -1.  Items
  // are also handed out once `stopped` is set: what a cancelled band leaves of
  // them is the caller's.
  __device__ __forceinline__ long long take(const BandBufs &b, int rank, int need) {
    const int have = (int)(end - cur < need ? end - cur : need);
    long long mine = rank < have ? cur + rank : -1;
    cur += have;
    if (have < need && !dry) {
      const long long left = n - end;
      const long long fair = left / (4ll * waves);
      const long long run = fair < need - have ? need - have : fair > max_run ? max_run : fair;
      unsigned long long base = 0;
      if (__lane_id() == 0) {
        base = atomicAdd(queue, (unsigned long long)run);
        if constexpr (Poll) {
          if (!(base & kStopBit) && crosses((long long)base, run, poll_shift) && poll_cancel(b, queue)) base |= kStopBit;
        }
      }
      base = first_lane(base);
      if constexpr (Poll) {
        stopped = (base & kStopBit) != 0;
        base &= kStopBit - 1;
      }
      const long long first = shared + (long long)base;
      cur = first + (need - have);
      end = first + run;
      if (end >= n) {
        dry = first >= n;
        end = n;
      }
      if (cur > end) cur = end;
      if (rank >= have && rank < need && first + (rank - have) < n) mine = first + (rank - have);
    }
    return mine;
  }
};

// The lanes of a wave over a queue of items, one distance estimate per lane
// and step (as k_march64 does with its rays): a lane is NEED (wants an item), ITER
// (its estimate is running), DONE (its estimate is complete, its item's next
// step pending) or EXHAUSTED.  fetch(rank, n): lanes in NEED take the items
// after the first n; step(): one formula iteration; done(): the item's next
// step.
template <int Iters, class Fetch, class Step, class Done>
__device__ __forceinline__ void lane_loop(int &state, Fetch fetch, Step step, Done done) {
  const int lane = __lane_id();
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (;;) {
    const unsigned long long m_need = __ballot(state == MS_NEED);
    const unsigned long long m_iter = __ballot(state == MS_ITER);
    const unsigned long long m_done = __ballot(state == MS_DONE);
    if (!(m_need | m_iter | m_done)) break;
    const int n_need = __popcll(m_need), n_iter = __popcll(m_iter), n_done = __popcll(m_done);
    if (n_need && (4 * n_need >= n_need + n_iter + n_done || n_iter + n_done == 0))
      fetch(__popcll(m_need & lt_mask), n_need);
    if (state == MS_ITER) {
      bool fin = false;
      for (int q = 0; q < Iters && !fin; q++) fin = step();
      if (fin) state = MS_DONE;
    }
    const unsigned long long m_done2 = __ballot(state == MS_DONE);
    const unsigned long long m_iter2 = __ballot(state == MS_ITER);
    const int n_done2 = __popcll(m_done2), n_iter2 = __popcll(m_iter2);
    if (n_done2 && (4 * n_done2 >= n_done2 + n_iter2 || n_iter2 == 0) && state == MS_DONE) done();
  }
}

// Workgroups of a kernel that fit the current device at once; `known` holds them
// per device (0: not asked yet), since devices may differ in their CUs.
constexpr int kKnownDevices = 32;
inline int resident_blocks(const void *kernel, std::atomic<int> (&known)[kKnownDevices]) {
  int dev = 0, per_cu = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 1 << 20;
  const bool keep = dev >= 0 && dev < kKnownDevices;
  int n = keep ? known[dev].load(std::memory_order_relaxed) : 0;
  if (n > 0) return n;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBlock, 0) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || per_cu * cus <= 0)
    return 1 << 20;
  n = per_cu * cus;
  if (keep) known[dev].store(n, std::memory_order_relaxed);
  return n;
}

// Launch of a persistent kernel: at most the workgroups that fit the chip at
// once (and `blocks`, the caller's share), so that no wave starts on its first
// items only after the others ran out.  (Where another stream's kernels hold
// the chip some still do.)
template <auto Kernel, class... A>
static void launch_resident(int blocks, hipStream_t s, A... args) {
  static std::atomic<int> known[kKnownDevices];
  const int resident = resident_blocks((const void *)Kernel, known);
  hipLaunchKernelGGL(Kernel, dim3((unsigned)std::max(1, std::min(blocks, resident))), dim3(kBlock), 0, s, args...);
}

}  // namespace mbr
