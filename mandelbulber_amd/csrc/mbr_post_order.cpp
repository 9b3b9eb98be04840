// mbr_post_order.cpp — host side of the depth-of-field post effect: the
// order in which PostRendering_DOF (src/image.cpp:57-247) splats its pixels.
//
// The reference sorts the zBuffer (QuickSortZBuffer, src/common_math.h:53-84,
// called on indices [1, n-1]) and then, from the far end, swaps each entry
// with a randomly drawn earlier one of similar blur size (image.cpp:96-152).
// Both steps are sequential and define the result (splats blend in this
// order), so they run here, on the host, exactly; the splatting itself runs
// on the GPU as an order-preserving gather (mbr_post.hip).
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <exception>
#include <thread>
#include <utility>
#include <vector>

#include "mbr_kernels.hpp"
#include "mbr_rand.hpp"

namespace mbr {

namespace {

struct ZEntry {
  float z;
  int i;
};

// Hoare partition of [l, p] around its middle element, ascending z; on return
// [l, j] and [i, p] are left to sort.
inline void zpartition(ZEntry *d, int l, int p, int &i_out, int &j_out) {
  int i = l, j = p;
  const float x = d[(l + p) / 2].z;
  do {
    while (d[i].z < x) i++;
    while (x < d[j].z) j--;
    if (i <= j) {
      const ZEntry t = d[i];
      d[i] = d[j];
      d[j] = t;
      i++;
      j--;
    }
  } while (i <= j);
  i_out = i;
  j_out = j;
}

// The two sides of a partition are independent ranges, so the order in which
// they are sorted does not change the result: the smaller sides of a range's
// first kForks partitions, where large, go to threads of their own (which fork
// again, each with the forks its parent has left: at most 2^kForks - 1 = 15
// threads in all), the larger side of the others to a stack (at most log2 n of
// them).  Without a thread to be had the range is sorted here.
constexpr int kForks = 4;
void zsort(ZEntry *d, int lo, int hi, int forks) {
  std::pair<int, int> stack[32];
  std::thread threads[kForks];
  int depth = 0, forked = 0;
  for (;;) {
    int i, j;
    zpartition(d, lo, hi, i, j);
    // sides of one entry (or none) are sorted
    std::pair<int, int> small{lo, j}, large{i, hi};
    if (small.second - small.first > large.second - large.first) std::swap(small, large);
    const bool more = small.first < small.second;
    if (more && forks > forked && small.second - small.first > 4096) {
      try {
        threads[forked] = std::thread(zsort, d, small.first, small.second, forks - forked - 1);
        forked++;
        lo = large.first;
        hi = large.second;
        continue;
      } catch (const std::exception &) {  // no thread, or no memory for its state
        forks = forked;
      }
    }
    if (more) {
      stack[depth++] = large;
      lo = small.first;
      hi = small.second;
    } else if (large.first < large.second) {
      lo = large.first;
      hi = large.second;
    } else if (depth > 0) {
      lo = stack[--depth].first;
      hi = stack[depth].second;
    } else {
      break;
    }
  }
  for (int k = 0; k < forked; k++) threads[k].join();
}

// Whether a pixel of blur size s2 may take the place of one of size s1
// (src/image.cpp:127-139): both on the same side of the focus and s2 / s1 (s1 /
// s2 in front of it) above 0.7.
inline bool similar(double s1, double s2) {
  if (!(s1 * s2 > 0)) return false;
  const double cmp = s1 > 0 ? s2 / s1 : s1 / s2;
  return cmp > 0.7;
}

}  // namespace

// The shuffle is a chain of random draws whose tests decide how many there are,
// so it stays on one thread, and its time is that of the mispredicted tests and
// of the reads behind them.  The tests read FP32 blur sizes, half the memory of
// the entries and no division, and go to the FP64 sizes only within 1e-5 of the
// bound (or beyond FP32's range); the draws come in blocks.  (Four candidates
// tested together without branches were slower, 21 against 13 ms for 480000
// pixels: each pixel's draws then wait for the last pixel's tests.)
void dof_order(const float *z, int width, int height, double neutral, double deep, uint32_t seed, uint32_t *rank) {
  const int n = width * height;
  std::vector<ZEntry> d((size_t)n);
  for (int k = 0; k < n; k++) d[k] = {z[k], k};
  if (n > 2) zsort(d.data(), 1, n - 1, kForks);
  auto size_of = [&](float zf) {
    const double zd = zf;
    return (zd - neutral) / zd * deep;
  };
  std::vector<float> blur((size_t)n);
  for (int k = 0; k < n; k++) blur[k] = (float)size_of(d[k].z);
  GlibcRand rnd(seed);
  uint32_t draws[GlibcRand::kBlock];
  int at = GlibcRand::kBlock;
  for (int i = n - 1; i >= 0; i--) {
    const float a = blur[i];
    const float lo = a * (a > 0 ? 0.69999f : 1.42858f), hi = a * (a > 0 ? 0.70001f : 1.42855f);
    const bool fast = std::fabs(a) > 1e-18f && std::fabs(a) < 1e18f;
    int step = i, ii;
    for (;;) {
      if (at == GlibcRand::kBlock) {
        rnd.block(draws);
        at = 0;
      }
      ii = i - (int)(draws[at++] % ((uint32_t)step + 1u));
      if (ii <= 0) ii = 0;
      const float b = blur[ii], m = std::fabs(b);
      // (the reference's "both sizes 0: done" is overwritten by this test)
      if (fast && (b > hi || b < lo) && m > 1e-18f && m < 1e18f) {
        if (b > hi && (a > 0 || b < 0)) break;
      } else if (similar(size_of(d[i].z), size_of(d[ii].z))) {
        break;
      }
      step = (int)(step * 0.7 - 1);
      if (step <= 0) break;
    }
    std::swap(d[i], d[ii]);
    blur[i] = blur[ii];
    blur[ii] = a;
  }
  // the splat loop runs from the end of the array
  for (int k = 0; k < n; k++) rank[d[(size_t)n - 1 - k].i] = (uint32_t)k;
}

}  // namespace mbr
