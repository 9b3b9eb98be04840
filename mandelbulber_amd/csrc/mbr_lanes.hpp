// mbr_lanes.hpp — how the persistent kernels share out their work: the queues
// that hand items to the lanes of a wave, the loop that keeps lanes busy with
// distance estimates of different lengths, and the launch of such a kernel.
#pragma once

#include <algorithm>

#include "mbr_kernels.hpp"

namespace mbr {

constexpr int kBlock = 256;

// A lane wants an item, runs an estimate, has an estimate complete, or found
// the queue empty.
enum : int { MS_NEED = 0, MS_ITER = 1, MS_DONE = 2, MS_EXHAUSTED = 3 };

// Cancel polling (mbr_cancel, the reference's programClosed test per pixel,
// src/Render3D.cpp:369-378).  take_work(queue, n) is the hand-out of a band
// work queue (lane 0 only): it returns the first of n items and whether the
// band was stopped.  A hand-out whose range crosses a multiple of
// 2^poll_shift reads the host flag (a read over the bus, so not on every
// hand-out); when set it adds kStopBit to the queue, so every later
// hand-out sees the stop in the value its own atomic returns.
constexpr unsigned long long kStopBit = 1ull << 48;

__device__ __forceinline__ unsigned long long take_work(const BandBufs &b, unsigned long long *queue,
                                                        unsigned long long n, int poll_shift, int &stopped) {
  unsigned long long v = atomicAdd(queue, n);
  if (b.cancel && !(v & kStopBit)) {
    const unsigned long long first = v & (kStopBit - 1);
    if (((first + n) >> poll_shift) != (first >> poll_shift) && *b.cancel != 0) {
      atomicAdd(queue, kStopBit);
      v |= kStopBit;
    }
  }
  stopped = (v & kStopBit) != 0;
  return v & (kStopBit - 1);
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
// and a run grows with what is left (up to 4 waves' worth, and so that every
// wave of the launch can still take 4 runs).
struct WaveQueue {
  unsigned long long *queue;
  long long n, cur, end, shared;  // shared: first item handed out by the counter
  int waves;
  bool dry, stopped;

  __device__ __forceinline__ WaveQueue(unsigned long long *queue_, long long n_, int lanes) {
    queue = queue_;
    n = n_;
    stopped = false;
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
  // For the whole wave: lane `rank` of `need` lanes gets its item, or -1.
  // Poll: the items are rays whose hand-out polls the cancel flag (take_work);
  // stop is then set once the band was stopped.
  template <bool Poll>
  __device__ __forceinline__ long long take(const BandBufs &b, int rank, int need, int poll_shift, int &stop) {
    const int have = (int)(end - cur < need ? end - cur : need);
    long long mine = rank < have ? cur + rank : -1;
    cur += have;
    if (have < need && !dry) {
      const long long left = n - end;
      const long long fair = left / (4ll * waves);
      const long long run = fair < need - have ? need - have : fair > 256 ? 256 : fair;
      unsigned long long base = 0;
      if (__lane_id() == 0) {
        if constexpr (Poll) base = take_work(b, queue, (unsigned long long)run, poll_shift, stop);
        else base = atomicAdd(queue, (unsigned long long)run);
      }
      base = __shfl(base, 0);
      if constexpr (Poll) stop = __shfl(stop, 0);
      const long long first = shared + (long long)base;
      cur = first + (need - have);
      end = first + run;
      if (end >= n) {
        dry = first >= n;
        end = n;
      }
      if (cur > end) cur = end;
      if (rank >= have && rank < need && first + (rank - have) < n) mine = first + (rank - have);
      if constexpr (Poll) stopped = stop != 0;
    }
    if constexpr (Poll) stop = stopped;
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


// Launch of a persistent kernel: at most the workgroups that fit the chip at
// once (and `blocks`, the caller's share), so that no wave starts on its first
// items only after the others ran out.
template <auto Kernel, class... A>
static void launch_resident(int blocks, hipStream_t s, A... args) {
  static const int resident = [] {
    int per_cu = 0, dev = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, Kernel, kBlock, 0) != hipSuccess ||
        hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || per_cu * cus <= 0)
      return 1 << 20;
    return per_cu * cus;
  }();
  hipLaunchKernelGGL(Kernel, dim3((unsigned)std::max(1, std::min(blocks, resident))), dim3(kBlock), 0, s, args...);
}

}  // namespace mbr
