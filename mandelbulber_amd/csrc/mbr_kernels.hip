// mbr_kernels.hip — gfx950 kernels of the render core.
//
// One frame (or band of rows) runs as these launches:
//   k_march64   one lane per primary ray: DE-stepped march with step records,
//               then the binary-search refinement, in FP64 (RayMarching,
//               src/Render3D.cpp:79-199); hits are appended to a compacted hit
//               list so shading runs on full waves of hits.  FP32_MARCH: k_march
//               in FP32 first, then k_march64 over the rays it handed over.
//   k_hits      shadow rays, normals (slowShading's: k_slow_normals) and colours
//               of the hits (ObjectShader, src/shaders.cpp:21); k_fast_ao or
//               k_ao their ambient occlusion, k_compose the sums.
//   k_finish    one lane per ray: background for misses, VolumetricShader
//               (glow, fog, volumetric fog) over the step record read back to
//               front, and coalesced writes of the framebuffer planes
//               (src/Render3D.cpp:530-589).
#include <type_traits>

#include "mbr_kernels.hpp"
#include "mbr_lanes.hpp"
#include "mbr_shade.hpp"

// This source is compiled once per unit of launches, in parallel (build.py);
// without MBR_PART it holds them all.
#ifdef MBR_PART
#define MBR_UNIT(k) (MBR_PART == (k))
#else
#define MBR_UNIT(k) 1
#endif

namespace mbr {

constexpr double kPi = 3.14159265358979323846;


// Step record writer of one ray: records below the slab size go to the
// step-major slab, later ones to chunks of the overflow pool listed in the
// ray's directory; the ray takes its directory (one atomic) on its first
// overflowing record and each chunk on the chunk's first record.  A
// re-march of the same ray reuses them.  When the pool is full the record
// is dropped and ST_POOL_MISS tells the host to grow the pool and render
// the band again.  All records of one ray are written by one lane.
constexpr unsigned long long kOneDir = 1ull << 32;
// fields of a lane's overflow count (misses: one bit)
constexpr unsigned long long kOvfRay = 1, kOvfChunk = 1ull << 20, kOvfMiss = 1ull << 44;
template <class RT>
struct RecPlanes {
  RT *step, *dist, *thr;     // slab planes
  RT *ostep, *odist, *othr;  // overflow pool planes
  int *it, *oit;             // iteration counts (null unless iteration fog is on)
  long long *ovf_off;
  int *dir;
  unsigned long long *pool;  // directories (times kOneDir) and chunks handed out
  long long cap, max_dirs, max_chunks;
  int slab, r;
  // ovf counts what the ray's lane adds to the overflow counters of the stats;
  // an add to a shared counter for each would serialise the waves
  __device__ __forceinline__ void put(int i, double step_v, double dist_v, double thr_v, int iters,
                                      unsigned long long &ovf) const {
    long long o;
    RT *st, *di, *th;
    int *itp;
    if (i < slab) {
      o = (long long)i * cap + r;
      st = step; di = dist; th = thr; itp = it;
    } else {
      long long dj = ovf_off[r];
      int first = -1;
      if (dj == -1) {
        // a directory and the first chunk with one add
        const unsigned long long n = atomicAdd(pool, kOneDir + 1);
        ovf += kOvfRay;
        dj = (long long)(n / kOneDir) < max_dirs ? (long long)(n / kOneDir) : -2;
        const long long ch = (long long)(n % kOneDir);
        first = ch < max_chunks ? (int)ch : -2;
        if (dj >= 0)
          for (int k = 0; k < kDirSlots; k++) dir[dj * kDirSlots + k] = -1;
        ovf_off[r] = dj;
      }
      if (dj < 0) {
        ovf |= kOvfMiss;
        return;
      }
      const int rel = i - slab;
      int *slot = &dir[dj * kDirSlots + rel / kChunk];
      int ch = first != -1 ? first : *slot;
      if (ch == -1) {
        const long long n = (long long)(atomicAdd(pool, 1ull) % kOneDir);
        ch = n < max_chunks ? (int)n : -2;
        first = ch;
      }
      if (first != -1) {
        ovf += kOvfChunk;
        *slot = ch;
      }
      if (ch < 0) {
        ovf |= kOvfMiss;
        return;
      }
      o = (long long)ch * kChunk + rel % kChunk;
      st = ostep; di = odist; th = othr; itp = oit;
    }
    st[o] = (RT)step_v;
    di[o] = (RT)dist_v;
    th[o] = (RT)thr_v;
    if (itp) itp[o] = iters;
  }
};

// The overflow counts of a lane into its stats.
__device__ __forceinline__ void add_ovf(unsigned long long (&v)[ST_COUNT], unsigned long long ovf) {
  v[ST_OVF_RAYS] = ovf % kOvfChunk;
  v[ST_OVF_CHUNKS] = ovf / kOvfChunk % (kOvfMiss / kOvfChunk);
  v[ST_POOL_MISS] = ovf / kOvfMiss;
}

// block-level reduction of per-lane counters into the device stats: LDS
// atomics inside the workgroup, then one global atomic per counter
__device__ __forceinline__ void flush_stats(unsigned long long *stats, const unsigned long long (&v)[ST_COUNT]) {
  __shared__ unsigned long long acc[ST_COUNT];
  if (threadIdx.x < ST_COUNT) acc[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ST_COUNT; i++)
    if (v[i]) atomicAdd(&acc[i], v[i]);
  __syncthreads();
  if (threadIdx.x < ST_COUNT && acc[threadIdx.x]) atomicAdd(&stats[threadIdx.x], acc[threadIdx.x]);
}

// ----------------------------------------------------------------- march
// The FP32 march (k_march) splits RayMarching (src/Render3D.cpp:79-199) around
// its distance estimates.  march_before_de sets up step i (point, threshold);
// march_after_de takes step i's distance and either continues, ends the ray
// as a miss, or hands the ray over to the FP64 continuation (k_march64).
//
// Hand-over rule.  A ray is handed over when step i's FP32 distance could be
// a hit once FP32 error is allowed for: below 1.001 x threshold, or within the
// drift margin of it.
//
// Drift model.  An FP32 distance differs from the FP64 distance at the same
// point by about 1e-6 of the distance (rounding accumulated over the
// iterations) plus the FP32 rounding of the point, 6e-8 of its largest
// coordinate; the step taken from it (times DE_factor) carries that error
// into the scan.  The errors of successive steps are independent roundings,
// so the scan's deviation from the FP64 march is estimated by their root sum
// of squares, sigma; the margin is 4 sigma.  The continuation decides every
// later hit test and every binary-search branch in FP64.  A decision that
// lies within the margin of its threshold may differ from the FP64 march's.
// Either way the binary search ends in the band where the distance lies in
// (thr (1 - 0.01 quality), thr), next to the point where the decision was
// taken; along the ray the distance changes at rate g (estimated from the
// last two distance estimates), so that band spans about
//   W = (0.01 quality thr + 2 margin) / g
// of depth, and both outcomes end within W of each other.  A branch whose
// step is below 5e-6 of the depth moves the result by less than 2e-5 of the
// depth and is not counted.  The ray is re-marched in FP64 from the start
// when a counted decision was ambiguous and W exceeds kRedoTol of the
// depth, i.e. on grazing incidence.
constexpr double kRedoTol = 3e-5;

struct MarchOut {
  V3<double> point;
  double scan, distThresh, dist;
  int buffCount, object;
  bool found;
};

struct RayState {
  V3<double> point;
  double scan, step, thr, drift, dist;
  double thr0;  // initial threshold: 0, or the previous ray's final one for a reflected ray
  int i, object;
};

enum : int { SO_CONTINUE = 0, SO_MISS = 1, SO_HANDOFF = 2 };

// What every step reads of the scene, held in registers: the kernels' stores
// keep the compiler from hoisting the loads out of their loops, and a step of a
// primary ray has fewer than two formula iterations to hide them behind.
struct MarchK {
  double resolution, persp, quality, DE_factor, far, below;
  int constant_thresh, wide, jitter;
};
__device__ __forceinline__ MarchK march_k(const DevScene &sc) {
  const ShadeK<double> &k = sc.sd;
  return MarchK{k.resolution, k.persp, k.quality, k.DE_factor, sc.view_distance_max, sc.interior ? 0.8 : 0.5,
                sc.constant_thresh, sc.persp_type == 1 || sc.persp_type == 2, sc.jitter_mode};
}

// The threshold at a distance along the ray; a quality of 1 needs no division.
// thr0: 0, or a reflected ray's initial threshold (distThreshInit,
// src/Render3D.cpp:92, :102-109).
__device__ __forceinline__ double march_thr(const MarchK &m, double scan, double thr0) {
#pragma clang fp contract(off)
  if (m.constant_thresh) return m.quality;
  double t = scan * m.resolution * m.persp;
  if (m.quality != 1.0) t = t / m.quality;
  return t + thr0;
}

__device__ __forceinline__ void march_before_de(const MarchK &m, V3<double> start, V3<double> dir, RayState &s) {
#pragma clang fp contract(off)
  s.point = start + dir * s.scan;
  s.thr = march_thr(m, s.scan, s.thr0);
  if (m.wide) s.thr *= kPi;
}

// obj_it: the estimate's object type in the low 3 bits, its iteration count
// (CalculateDistance's itersOut) above them.
__device__ __forceinline__ int march_after_de(const MarchK &m, RayState &s, double d, int obj_it, uint32_t ray_hash,
                                              const RecPlanes<float> &rec, unsigned long long &ovf) {
#pragma clang fp contract(off)
  s.object = obj_it & 7;
  const double dist = d > 3.0 ? 3.0 : d;
  // s.drift holds the variance of the scan deviation
  const double pmax = fmax(fabs(s.point.x), fmax(fabs(s.point.y), fabs(s.point.z)));
  const double err = 1e-6 * fabs(d) + 6e-8 * pmax;
  if (dist < 1.001 * s.thr || dist - s.thr < 4.0 * sqrt(s.drift + err * err)) return SO_HANDOFF;
  const double jf = m.jitter ? jitter_factor(jitter_draw(ray_hash, (uint32_t)s.i)) : 1.0;
  const double old_step = s.step;
  s.step = (dist - m.below * s.thr) * m.DE_factor * jf;
  rec.put(s.i, old_step, d, s.thr, obj_it >> 3, ovf);
  s.scan += s.step;
  s.drift += (err * m.DE_factor) * (err * m.DE_factor);
  s.dist = dist;
  s.i++;
  if (s.scan > m.far || s.i >= 10000) return SO_MISS;
  return SO_CONTINUE;
}

__device__ __forceinline__ RayState ray_start_state(const DevScene &sc) {
  RayState s;
  s.point = v3<double>(0, 0, 0);
  s.scan = sc.view_distance_min;
  s.step = sc.view_distance_min;
  s.thr = 0.0;
  s.thr0 = 0.0;
  s.drift = 0.0;
  s.dist = 0.0;
  s.i = 0;
  s.object = OBJ_FRACTAL;
  return s;
}

// The result of a ray's march.
__device__ __forceinline__ void write_ray(const BandBufs &b, int r, const MarchOut &o) {
  b.found[r] = o.found;
  b.object[r] = (uint8_t)o.object;
  b.count[r] = o.buffCount;
  b.depth[r] = o.scan;
  b.thr[r] = o.distThresh;
  b.last[r] = o.dist;
  b.px[r] = o.point.x;
  b.py[r] = o.point.y;
  b.pz[r] = o.point.z;
}

// Appends to one of the band's lists (hits, hand-overs, redos) through a buffer
// of the wave in LDS, 64 entries per add to the list's counter: adds to one
// address pass at about 13 ns each, so one add per hit-finding step block held
// a 4K frame's march for several ms.  Lists have no order.
struct WaveListBuf {
  int entry[kBlock / 64][128];
  int count[kBlock / 64];
};
struct WaveList {
  WaveListBuf &buf;

  __device__ __forceinline__ explicit WaveList(WaveListBuf &buf_) : buf(buf_) {
    buf.count[threadIdx.x >> 6] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  // by any lanes
  __device__ __forceinline__ void append(int r) {
    const int w = (int)(threadIdx.x >> 6);
    buf.entry[w][atomicAdd(&buf.count[w], 1)] = r;
  }
  // by the whole wave, after at most one append per lane; all: to the last entry
  __device__ __forceinline__ void flush(int *out, unsigned long long *counter, bool all) {
    const int lane = __lane_id(), w = (int)(threadIdx.x >> 6);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    int n = __builtin_amdgcn_readfirstlane(buf.count[w]);
    while (n >= 64 || (all && n > 0)) {
      const int m = n < 64 ? n : 64;
      unsigned long long base = 0;
      if (lane == 0) base = atomicAdd(counter, (unsigned long long)m);
      base = __shfl(base, 0);
      if (lane < m) out[base + lane] = buf.entry[w][lane];
      const int rest = 64 + lane < n ? buf.entry[w][64 + lane] : 0;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (64 + lane < n) buf.entry[w][lane] = rest;
      n -= m;
      buf.count[w] = n;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
};

template <class RT>
__device__ __forceinline__ RecPlanes<RT> ray_records(const BandBufs &b, int r) {
  RecPlanes<RT> rec;
  rec.step = (RT *)b.rec_step;
  rec.dist = (RT *)b.rec_dist;
  rec.thr = (RT *)b.rec_thr;
  rec.ostep = (RT *)b.ovf_step;
  rec.odist = (RT *)b.ovf_dist;
  rec.othr = (RT *)b.ovf_thr;
  rec.it = b.rec_it;
  rec.oit = b.ovf_it;
  rec.ovf_off = b.ovf_off;
  rec.dir = b.ovf_dir;
  rec.pool = &b.counters[CNT_POOL];
  rec.cap = b.cap;
  rec.max_dirs = b.ovf_dirs;
  rec.max_chunks = b.ovf_chunks;
  rec.slab = b.slab;
  rec.r = r;
  return rec;
}

// Whether a kernel of formula F keeps a copy of the scene's formula constants.
// The plain variants read a few of them in every iteration, and the stores and
// atomics of the loops keep the compiler from hoisting loads of the scene block:
// a local copy keeps them in registers.  Not where the scene may rotate (the
// Mandelbox's 13 matrices) or fold nine times (the kaleidoscopic IFS): their
// copies are spilled and read back lane by lane, which cost 1.9 times the time
// of the rotated Mandelbox's FP64 AO (480x320, 8.0 and 15.2 ms).
constexpr bool local_scene(int F, int P) { return P && F != 10 && !(F == 8 && P == kPlain); }

// Persistent march: one primary ray per lane, up to kMarchIters formula
// iterations per pass, lane states and amortised bookkeeping as in k_ao.
#ifndef MBR_MARCH_ITERS
#define MBR_MARCH_ITERS 6
#endif
constexpr int kMarchIters = MBR_MARCH_ITERS;
// hand-outs poll the cancel flag every 2^kPollRays rays of the march and every
// 2^kPollHits hits of AO
constexpr int kPollRays = 12, kPollHits = 8;
// and a wave takes that many rays, or hits of that many AO directions, with one add
constexpr int kRayRun = 128;
constexpr unsigned kRunDirs = 2048;

// IP: the integer power of the Mandelbulb when fixed at compile time (8).
template <int F, int Plain, int IP>
__device__ __forceinline__ void march_body(const DevScene *__restrict__ scp, BandBufs b, int band_first,
                                           int band_rays, unsigned long long *stats) {
  using T = float;
  using RT = float;
  // integer-power Mandelbulb iterations without inverse trig wherever the
  // records are FP32; the FP64 mode keeps the trigonometric form
  constexpr bool kAlg = sizeof(RT) < 8 || IP != 0;
  const DevScene &sc = *scp;
  constexpr bool kLocal = local_scene(F, Plain);
  const FractalK<T> f_local = kLocal ? sc.frac<T>() : FractalK<T>{};
  const FractalK<T> &f = kLocal ? f_local : sc.frac<T>();
  const int N = sc.N, minN = sc.minN;
  const int lane = __lane_id();
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const V3<double> start = v3<double>(sc.start[0], sc.start[1], sc.start[2]);

  const MarchK m = march_k(sc);
  __shared__ WaveListBuf hand_buf;
  WaveList hand(hand_buf);
  const int lanes = item_lanes(band_rays);
  WaveQueue<true> q(&b.counters[CNT_RAYQ], band_rays, lanes, kRayRun, kPollRays);
  int state = lane < lanes ? MS_NEED : MS_EXHAUSTED;
  int r = 0;
  uint32_t ray_hash = 0;
  V3<double> dir = v3<double>(0, 0, 0);
  RayState s = ray_start_state(sc);
  DECall<T> call;
  T dist = 0;
  int object = OBJ_FRACTAL;
  bool early = false;  // the estimate ended in begin_de, without iterating
  LaneCount cnt = {0, 0};
  unsigned long long ovf = 0;

  auto begin_de = [&]() {
    march_before_de(m, start, dir, s);
    DEInfo info;
    const V3<T> p = cvt<T>(s.point);
    early = de_call_begin<T, F, Plain, kAlg, IP>(f, p, (T)s.thr, N, minN, false, call, dist, info);
    state = early ? MS_DONE : MS_ITER;
    if (early) object = info.object | (info.iters << 3);
  };

  for (;;) {
    const unsigned long long m_need = __ballot(state == MS_NEED);
    const unsigned long long m_iter = __ballot(state == MS_ITER);
    const unsigned long long m_done = __ballot(state == MS_DONE);
    if (!(m_need | m_iter | m_done)) break;
    const int n_need = __popcll(m_need), n_iter = __popcll(m_iter), n_done = __popcll(m_done);

    if (n_need && (4 * n_need >= n_need + n_iter + n_done || n_iter + n_done == 0)) {
      const long long mine = q.take(b, __popcll(m_need & lt_mask), n_need);
      if (state == MS_NEED) {
        if (mine < 0) {
          state = MS_EXHAUSTED;
        } else {
          r = (int)mine;
          b.ovf_off[r] = -1;
          const int p = band_first + r;
          const int x = p % sc.width, y = p / sc.width;
          // a cancelled band's remaining rays take the empty record of a
          // cut ray, so later kernels read defined (if meaningless) values
          const bool cut = q.stopped || view_vector(sc, x, y, dir);
          ray_hash = jitter_ray(sc.jitter_seed, sc.frame_no, sc.pixel_base + (uint32_t)p);
          s = ray_start_state(sc);
          if (cut) {
            MarchOut o;
            o.point = v3<double>(0, 0, 0);
            o.scan = 0; o.distThresh = 0; o.dist = 0; o.buffCount = 0; o.object = OBJ_FRACTAL;
            o.found = false;
            write_ray(b, r, o);
          } else {
            begin_de();
          }
        }
      }
    }

    if (state == MS_ITER) {
      bool fin = false;
#pragma unroll
      for (int k = 0; k < kMarchIters && !fin; k++) fin = de_call_step<T, F, Plain, kAlg, IP>(f, call, N);
      if (fin) state = MS_DONE;
    }

    const unsigned long long m_done2 = __ballot(state == MS_DONE);
    const unsigned long long m_iter2 = __ballot(state == MS_ITER);
    bool appended = false;
    const int n_done2 = __popcll(m_done2), n_iter2 = __popcll(m_iter2);
    if (n_done2 && (4 * n_done2 >= n_done2 + n_iter2 || n_iter2 == 0) && state == MS_DONE) {
      cnt.de_calls += 1;
      if (!early) {
        DEInfo info;
        dist = de_call_end<T, F, Plain, kAlg, IP>(f, call, (T)s.thr, N, minN, false, info);
        object = info.object | (info.iters << 3);
        cnt.iterations += (uint32_t)info.work;
      }
      const int out = march_after_de(m, s, (double)dist, object, ray_hash, ray_records<RT>(b, r), ovf);
      if (out == SO_CONTINUE) {
        begin_de();
      } else if (out == SO_MISS) {
        MarchOut o;
        o.point = s.point;
        o.scan = s.scan;
        o.distThresh = s.thr;
        o.dist = s.dist;
        o.buffCount = s.i;
        o.object = s.object;
        o.found = false;
        write_ray(b, r, o);
        state = MS_NEED;
      } else {
        hand.append(r);
        b.hand_i[r] = s.i;
        b.hand_scan[r] = s.scan;
        b.hand_step[r] = s.step;
        b.hand_drift[r] = s.drift;
        b.hand_dist[r] = s.dist;
        appended = true;
        state = MS_NEED;
      }
    }
    if (__ballot(appended)) hand.flush(b.hand_ray, &b.counters[CNT_HAND], false);
  }
  hand.flush(b.hand_ray, &b.counters[CNT_HAND], true);
  unsigned long long v[ST_COUNT] = {0};
  add_ovf(v, ovf);
  v[ST_MARCH_DE] = cnt.de_calls;
  v[ST_MARCH_ITERS] = cnt.iterations;
  flush_stats(stats, v);
}

template <int F, int Plain, int IP>
__global__ void __launch_bounds__(kBlock) k_march(const DevScene *__restrict__ scp, BandBufs b, int band_first,
                                                  int band_rays, unsigned long long *stats) {
  march_body<F, Plain, IP>(scp, b, band_first, band_rays, stats);
}


// ---------------------------------------------------------- FP64 march
// RayMarching (src/Render3D.cpp:79-199) in FP64, march, binary search and
// (hit_refine) root refinement, one ray per lane and one distance estimate
// at a time: every lane is in one phase of its own ray, and when its estimate
// completes the phase's rule picks the next point or ends the ray, so lanes of
// one wave march, search and start new rays side by side.
//
// One kernel for all FP64 rays.  As two kernels (march, then a lane-per-ray
// loop over the hits for the search) the search took as long as its slowest
// lane per wave at 25-30% active lanes and 256 registers with up to 1500 bytes
// of scratch, ran every hit's last estimate twice, and a frame waited for the
// slowest ray of each kernel in turn.
//   kRays  the band's primary rays from their start (FP64 march modes)
//   kHand  rays the FP32 march handed over, from the step it stopped at; those
//          whose result FP32 error could have changed are listed for kRedo
//   kRedo  the listed rays from their start
//   kRefl  a reflection level's rays, each with its own start and threshold
enum : int { kRays = 0, kHand = 1, kRedo = 2, kRefl = 3 };
enum : int { PH_MARCH = 0, PH_SEARCH = 1, PH_PLUS = 2, PH_MINUS = 3, PH_ROOT = 4 };

// IP: the integer power of the Mandelbulb when fixed at compile time (8).
template <class RT, int F, int Plain, int IP, int Src>
__device__ __forceinline__ void march64_body(const DevScene *__restrict__ scp, BandBufs b, int band_first,
                                             int band_rays, unsigned long long *stats) {
#pragma clang fp contract(off)
  // integer-power Mandelbulb iterations without inverse trig wherever the
  // records are FP32; the FP64 mode keeps the trigonometric form
  constexpr bool kAlg = sizeof(RT) < 8 || IP != 0;
  const DevScene &sc = *scp;
  constexpr bool kLocal = local_scene(F, Plain);
  const FractalK<double> f_local = kLocal ? sc.fd : FractalK<double>{};
  const FractalK<double> &f = kLocal ? f_local : sc.fd;
  const MarchK m = march_k(sc);
  const int N = sc.N, minN = sc.minN;
  const int lane = __lane_id();
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const long long n_items = Src == kRays ? (long long)band_rays
                                         : (long long)b.counters[Src == kRedo ? CNT_REDO : CNT_HAND];
  __shared__ WaveListBuf hit_buf, redo_buf;  // (the latter's space is kHand's only)
  WaveList hit_list(hit_buf);
  WaveList redo_list(Src == kHand ? redo_buf : hit_buf);
  bool appended = false;
  const int lanes = item_lanes(n_items);
  WaveQueue<Src == kRays> q(&b.counters[Src == kRays ? CNT_RAYQ : Src == kRedo ? CNT_REDOQ : CNT_HANDQ], n_items, lanes,
                            kRayRun, kPollRays);
  const double search_limit = 1.0 - 0.01 * m.quality;
  const bool hit_refine = sc.hit_refine != 0;
  const double c0 = 1.0 - 0.005 * m.quality;
  const double kthr = m.resolution * m.persp / m.quality;

  int state = lane < lanes ? MS_NEED : MS_EXHAUSTED;
  int phase = PH_MARCH;
  int r = 0, j = 0;
  uint32_t ray_hash = 0;
  V3<double> start = v3<double>(sc.start[0], sc.start[1], sc.start[2]);
  V3<double> dir = v3<double>(0, 0, 0);
  RayState s = ray_start_state(sc);
  DECall<double> call;
  // the estimate, the threshold of the search, its step (the refinement: the
  // estimate ahead of the root)
  double dist = 0, thr = 0, step = 0;
  double prev_dist = 0, prev_scan = 0, margin = 0;
  bool early = false, ambiguous = false, have_prev = false, below = false;
  int early_obj = 0;  // object and iterations << 3 of an early estimate
  LaneCount cnt = {0, 0};
  unsigned long long ovf = 0;
  unsigned long long hits = 0, missed = 0, redo = 0;

  // start the estimate at distance t along the ray (detail size s.thr)
  auto begin_de = [&](double t) {
#pragma clang fp contract(off)
    const V3<double> p = start + dir * t;
    if constexpr (F == 0) {  // whole estimates: one call for all lanes, in the pass
      call.p = p;
      early = true;
      state = MS_ITER;
      return;
    }
    DEInfo info;
    early = de_call_begin<double, F, Plain, kAlg, IP>(f, p, s.thr, N, minN, false, call, dist, info);
    state = early ? MS_DONE : MS_ITER;
    if (early) {
      early_obj = info.object | (info.iters << 3);
      cnt.iterations += (uint32_t)info.work;
    }
  };
  // step s.i of the march
  auto begin_march = [&]() {
#pragma clang fp contract(off)
    s.thr = march_thr(m, s.scan, s.thr0);
    if (m.wide) s.thr *= kPi;
    thr = s.thr;
    phase = PH_MARCH;
    begin_de(s.scan);
  };
  // the ray's end; at: its last estimate
  auto finish = [&](bool found, double at) {
#pragma clang fp contract(off)
    if (Src == kHand && ambiguous) {
      // marched again from the start (kRedo)
      redo_list.append(r);
      appended = true;
      redo++;
      state = MS_NEED;
      return;
    }
    MarchOut o;
    o.point = start + dir * at;
    o.scan = s.scan;
    o.distThresh = thr;
    o.dist = found ? dist : s.dist;
    o.buffCount = s.i;
    o.object = s.object;
    o.found = found;
    write_ray(b, r, o);
    if (found) hit_list.append(r);
    appended |= found;
    hits += found;
    missed += found && below;
    state = MS_NEED;
  };
  // The next point of the binary search from the estimate `dist` at s.scan,
  // or true at its end (src/Render3D.cpp:163-183).
  auto search = [&]() -> bool {
#pragma clang fp contract(off)
    bool end = j >= 20;
    if (!end) {
      if constexpr (Src == kHand) {
        if (step > 5e-6 * s.scan && (fabs(dist - thr) < margin || fabs(dist - thr * search_limit) < margin))
          ambiguous = true;
      }
      end = dist < thr && dist > thr * search_limit;
    }
    if (!end) {
      if constexpr (Src == kHand) {
        prev_dist = dist;
        prev_scan = s.scan;
        have_prev = true;
      }
      if (dist > thr) s.scan += step;
      else if (dist < thr * search_limit) s.scan -= step;
      thr = march_thr(m, s.scan, s.thr0);
      step *= 0.5;
      j++;
      phase = PH_SEARCH;
      begin_de(s.scan);
      return false;
    }
    if constexpr (Src == kHand) {
      if (ambiguous && have_prev) {
        const double g = fabs(dist - prev_dist) / fmax(fabs(s.scan - prev_scan), 1e-300);
        const double W = (0.01 * m.quality * thr + 2.0 * margin) / fmax(g, 1e-12);
        ambiguous = W > kRedoTol * s.scan;
      }
    }
    j = 0;
    return true;
  };
  // Newton steps on F(t) = dist(t) - c0 thr(t), c0 the middle of the band,
  // with a central-difference slope; each step at most one threshold long; true when settled
  auto refine = [&]() -> bool {
#pragma clang fp contract(off)
    const double f0 = dist - c0 * kthr * s.scan;
    if (j < 8 && fabs(f0) > 1e-13 * kthr * s.scan) {
      const double eps = 1e-3 * kthr * s.scan;
      prev_dist = dist;
      phase = PH_PLUS;
      begin_de(s.scan + eps);
      return false;
    }
    thr = s.scan * kthr;
    return true;
  };

  for (;;) {
    const unsigned long long m_need = __ballot(state == MS_NEED);
    const unsigned long long m_iter = __ballot(state == MS_ITER);
    const unsigned long long m_done = __ballot(state == MS_DONE);
    if (!(m_need | m_iter | m_done)) break;
    const int n_need = __popcll(m_need), n_iter = __popcll(m_iter), n_done = __popcll(m_done);

    if (n_need && (F == 0 || 4 * n_need >= n_need + n_iter + n_done || n_iter + n_done == 0)) {
      const long long mine = q.take(b, __popcll(m_need & lt_mask), n_need);
      if (state == MS_NEED) {
        if (mine < 0) {
          state = MS_EXHAUSTED;
        } else {
          r = Src == kRays ? (int)mine : Src == kRedo ? b.redo_list[mine] : b.hand_ray[mine];
          s = ray_start_state(sc);
          ray_hash = jitter_ray(sc.jitter_seed, sc.frame_no, sc.pixel_base + (uint32_t)(band_first + r));
          bool cut_ray = false;
          if constexpr (Src == kRefl) {
            b.ovf_off[r] = -1;
            start = v3<double>(b.ray_o[3 * (long long)r], b.ray_o[3 * (long long)r + 1], b.ray_o[3 * (long long)r + 2]);
            dir = v3<double>(b.ray_d[3 * (long long)r], b.ray_d[3 * (long long)r + 1], b.ray_d[3 * (long long)r + 2]);
            s.thr0 = b.ray_t0[r];
          } else {
            const int p = band_first + r;
            // a cancelled band's remaining rays take the empty record of a
            // cut ray, so later kernels read defined (if meaningless) values
            cut_ray = view_vector(sc, p % sc.width, p / sc.width, dir);
            if constexpr (Src == kRays) {
              b.ovf_off[r] = -1;
              cut_ray = cut_ray || q.stopped;
            } else {
              cut_ray = false;  // the march handed it over
            }
          }
          if constexpr (Src == kHand) {
            s.i = b.hand_i[r];
            s.scan = b.hand_scan[r];
            s.step = b.hand_step[r];
            s.drift = b.hand_drift[r];
            s.dist = b.hand_dist[r];
            margin = 4.0 * sqrt(s.drift);  // s.drift: variance of the FP32 scan deviation
            prev_dist = s.dist;
            prev_scan = s.scan - s.step;  // the step before s.i
            have_prev = s.i > 0;
            ambiguous = false;
          }
          if (cut_ray) {
            MarchOut o;
            o.point = v3<double>(0, 0, 0);
            o.scan = 0; o.distThresh = 0; o.dist = 0; o.buffCount = 0; o.object = OBJ_FRACTAL;
            o.found = false;
            write_ray(b, r, o);
          } else {
            begin_march();
          }
        }
      }
    }

    if (state == MS_ITER) {
      bool fin = F == 0;
      if constexpr (F == 0) {
        DEInfo info;
        dist = calc_distance_generic<double, Plain>(f, call.p, s.thr, N, minN, false, info);
        early_obj = info.object | (info.iters << 3);
        cnt.iterations += (uint32_t)info.work;
      } else {
#pragma unroll
        for (int it = 0; it < kMarchIters && !fin; it++) fin = de_call_step<double, F, Plain, kAlg, IP>(f, call, N);
      }
      if (fin) state = MS_DONE;
    }

    const unsigned long long m_done2 = __ballot(state == MS_DONE);
    const unsigned long long m_iter2 = __ballot(state == MS_ITER);
    const int n_done2 = __popcll(m_done2), n_iter2 = __popcll(m_iter2);
    if (n_done2 && (4 * n_done2 >= n_done2 + n_iter2 || n_iter2 == 0) && state == MS_DONE) {
      int obj_it = early_obj;
      if (!early) {
        DEInfo info;
        dist = de_call_end<double, F, Plain, kAlg, IP>(f, call, s.thr, N, minN, false, info);
        obj_it = info.object | (info.iters << 3);
        cnt.iterations += (uint32_t)info.work;
      }
      cnt.de_calls += 1;
      bool found = false, settled = false;
      if (phase != PH_PLUS && phase != PH_MINUS) s.object = obj_it & 7;
      if (phase == PH_MARCH) {
        const double raw = dist;
        if (dist > 3.0) dist = 3.0;
        if constexpr (Src == kHand) {
          if (fabs(dist - s.thr) < margin) ambiguous = true;
        }
        if (dist < s.thr) {
          if constexpr (Src == kRays) {
            // mbr_stats.march_de_calls counts it for the march and for the search
            // that starts from it; it runs once, and its iterations count once
            cnt.de_calls += 1;
          }
          below = dist < 0.1 * s.thr;
          step = s.step * 0.5;
          j = 0;
          found = search();
        } else {
          const double jf = m.jitter ? jitter_factor(jitter_draw(ray_hash, (uint32_t)s.i)) : 1.0;
          const double old_step = s.step;
          s.step = (dist - m.below * s.thr) * m.DE_factor * jf;
          ray_records<RT>(b, r).put(s.i, old_step, raw, s.thr, obj_it >> 3, ovf);
          if constexpr (Src == kHand) {
            prev_dist = dist;
            prev_scan = s.scan;
            have_prev = true;
          }
          const double at = s.scan;
          s.scan += s.step;
          s.dist = dist;
          s.i++;
          if (s.scan > m.far || s.i >= 10000) finish(false, at);
          else begin_march();
        }
      } else if (phase == PH_SEARCH) {
        found = search();
      } else if (phase == PH_PLUS) {
        step = dist;
        phase = PH_MINUS;
        const double eps = 1e-3 * kthr * s.scan;
        begin_de(s.scan - eps);
      } else if (phase == PH_MINUS) {
        const double eps = 1e-3 * kthr * s.scan;
        const double g = (step - dist) / (2.0 * eps) - c0 * kthr;
        const double f0 = prev_dist - c0 * kthr * s.scan;
        if (!(fabs(g) > 0.0)) {
          dist = prev_dist;
          thr = s.scan * kthr;
          settled = true;
        } else {
          double dt = -f0 / g;
          const double lim = kthr * s.scan;
          dt = dt > lim ? lim : (dt < -lim ? -lim : dt);
          s.scan += dt;
          j++;
          phase = PH_ROOT;
          begin_de(s.scan);
        }
      } else {
        settled = refine();
      }
      if (found) settled = hit_refine && !m.constant_thresh ? refine() : true;
      if (settled) finish(true, s.scan);
    }
    if (__ballot(appended)) {
      hit_list.flush(b.hit_list, &b.counters[CNT_HITS], false);
      if constexpr (Src == kHand) redo_list.flush(b.redo_list, &b.counters[CNT_REDO], false);
      appended = false;
    }
  }
  hit_list.flush(b.hit_list, &b.counters[CNT_HITS], true);
  if constexpr (Src == kHand) redo_list.flush(b.redo_list, &b.counters[CNT_REDO], true);
  unsigned long long v[ST_COUNT] = {0};
  add_ovf(v, ovf);
  v[ST_MARCH_DE] = cnt.de_calls;
  v[ST_MARCH_ITERS] = cnt.iterations;
  v[ST_HITS] = hits;
  v[ST_MISSED] = missed;
  v[ST_REDO] = redo;
  flush_stats(stats, v);
}

template <class RT, int F, int Plain, int IP, int Src>
__global__ void __launch_bounds__(kBlock, !Plain ? 1 : (F == 2 && !IP) || F == 1 ? 2 : 4)
    k_march64(const DevScene *__restrict__ scp, BandBufs b, int band_first, int band_rays,
              unsigned long long *stats) {
  march64_body<RT, F, Plain, IP, Src>(scp, b, band_first, band_rays, stats);
}

template <class T>
struct SurfBufs {
  T *base;    // [3][n] mainLight * shade * shadow
  T *spec;    // [3][n] mainLight * specular * shadow
  T *col;     // [3][n] surface colour
  T *fast_ao; // [n]
  T *ao;      // [n * dirs] AO intensity per (hit, direction)
  T *aux;     // [6][n] aux lights: diffuse R, G, B, specular R, G, B
  long long n;
  double *est[4];  // k_hits: the normals' FP64 estimates of FP32 shading (the
                   // hand-over planes: these formulas' rays are not handed over)
  int fast_items;  // fast AO: estimates per hit, kept in ao ([i][hits]); 0: summed by k_fast_ao
};

template <class T>
__device__ __forceinline__ void load_hit(const DevScene &sc, const BandBufs &b, int r, ShaderIn<T> &in) {
  const ShadeK<T> &k = sc.shade<T>();
  in.point64 = v3<double>(b.px[r], b.py[r], b.pz[r]);
  in.point = cvt<T>(in.point64);
  in.light = v3<T>(k.light[0], k.light[1], k.light[2]);
  in.dist_thresh = (T)b.thr[r];
  in.lastDist = (T)b.last[r];
  in.depth = (T)b.depth[r];
  in.delta = sc.constant_thresh ? (T)(b.depth[r] * sc.sd.resolution * sc.sd.persp) : (T)(b.thr[r] * sc.sd.quality);
  in.detail = in.dist_thresh;
  in.object = b.object[r];
}

// The direction of ray r: the camera's view vector, or the mirrored
// direction of a reflection level.
__device__ __forceinline__ V3<double> ray_dir(const DevScene &sc, const BandBufs &b, int band_first, int r) {
  V3<double> dir;
  if (b.ray_d) {
    dir = v3<double>(b.ray_d[3 * (long long)r + 0], b.ray_d[3 * (long long)r + 1], b.ray_d[3 * (long long)r + 2]);
  } else {
    const int p = band_first + r;
    view_vector(sc, p % sc.width, p / sc.width, dir);
  }
  return dir;
}

// Writes the hit's colour planes and its 8-bit colour.
template <class T>
__device__ __forceinline__ void put_colour(const BandBufs &b, const SurfBufs<T> &sb, int r, long long tid,
                                           RGBT<T> colour) {
  const long long n = sb.n;
  sb.col[0 * n + tid] = colour.R;
  sb.col[1 * n + tid] = colour.G;
  sb.col[2 * n + tid] = colour.B;
  b.col_r[r] = x86_d2u8((double)colour.R * 255);
  b.col_g[r] = x86_d2u8((double)colour.G * 255);
  b.col_b[r] = x86_d2u8((double)colour.B * 255);
}

// ObjectShader's diffuse and specular terms of the main light from the hit's
// normal and shadow.
template <class T>
struct Lit {
  T base[3], spec[3];
};
template <class T>
__device__ __forceinline__ Lit<T> light_hit(const DevScene &sc, const ShaderIn<T> &in, T shadow) {
  const ShadeK<T> &k = sc.shade<T>();
  Lit<T> o;
  T sh = dot(in.normal, in.light);
  if (sh < 0) sh = 0;
  const T shade = k.direct_light * ((T(1) - k.shading) + k.shading * sh);
  V3<T> half = normalize(in.light - in.view);
  T shade2 = dot(in.normal, half);
  if (shade2 < T(0)) shade2 = 0;
  shade2 = Math<T>::pow(shade2, T(30));
  if (shade2 > T(15)) shade2 = 15;
  const T specular = shade2 * k.specular;
  for (int c = 0; c < 3; c++) {
    o.base[c] = k.main_light[c] * shade * shadow;
    o.spec[c] = k.main_light[c] * specular * shadow;
  }
  return o;
}

// Stores them, and what the later shaders read of the hit.
template <class T>
__device__ __forceinline__ void put_lit(const DevScene &sc, const ShaderIn<T> &in, const Lit<T> &o, long long tid,
                                        const SurfBufs<T> &sb) {
  const long long n = sb.n;
  for (int c = 0; c < 3; c++) {
    sb.base[c * n + tid] = o.base[c];
    sb.spec[c * n + tid] = o.spec[c];
  }
  if constexpr (sizeof(T) == 8) {
    if (sc.env_map) {
      // environment mapping x reflect (ObjectShader, src/shaders.cpp:73-80);
      // k_compose multiplies it by the AO
      double e[3];
      env_mapping(sc, cvt<double>(in.normal), cvt<double>(in.view), e);
      for (int c = 0; c < 3; c++) sb.aux[(6 + c) * n + tid] = (T)(e[c] * sc.reflect);
    }
  }
  if (sc.n_lights > 0 || sc.fake_lights) {
    // k_aux shades the aux (and fake) lights from the normal and the
    // detail size MainShadow left (the aux shadows inherit it)
    sb.aux[0 * n + tid] = in.normal.x;
    sb.aux[1 * n + tid] = in.normal.y;
    sb.aux[2 * n + tid] = in.normal.z;
    sb.aux[3 * n + tid] = in.detail;
  }
}

// A cancel during the march or the surface shading stops AO before its first
// hit (by one lane of the surface kernel, at the end of its items).
__device__ __forceinline__ void poll_before_ao(const DevScene &sc, const BandBufs &b) {
  if (sc.ao && !sc.fast_ao && blockIdx.x == 0 && threadIdx.x == 0) poll_cancel(b, &b.counters[CNT_AOQ]);
}

// The generic formulas' surface shading (of trig_DE and the kaleidoscopic IFS:
// in scenes that are not plain), one lane per hit (their estimates
// run whole, so there is nothing to interleave).
template <class T>
__global__ void __launch_bounds__(kBlock) k_surface_generic(const DevScene *__restrict__ scp, BandBufs b,
                                                            int band_first, SurfBufs<T> sb,
                                                            unsigned long long *stats) {
  const DevScene &sc = *scp;
  const long long n_hits = (long long)b.counters[CNT_HITS];
  LaneCount cnt = {0, 0};
  for (long long tid = (long long)blockIdx.x * kBlock + threadIdx.x; tid < n_hits;
       tid += (long long)gridDim.x * kBlock) {
    const int r = b.hit_list[tid];
    ShaderIn<T> in;
    load_hit(sc, b, r, in);
    in.view = cvt<T>(ray_dir(sc, b, band_first, r));
    in.normal = normals<T, 0>(sc, in, cnt);
    T shadow = 1;
    if (sc.shadow) shadow = main_shadow<T, 0>(sc, in, cnt);
    const RGBT<T> colour = surface_colour<T, false, true>(sc, in, cnt);
    put_lit<T>(sc, in, light_hit<T>(sc, in, shadow), tid, sb);
    put_colour(b, sb, r, tid, colour);
    if (sc.ao && sc.fast_ao) sb.fast_ao[tid] = fast_ao2<T, 0>(sc, in, cnt);
    else if (sc.ao) sb.fast_ao[tid] = in.detail;
  }
  poll_before_ao(sc, b);
  unsigned long long v[ST_COUNT] = {0};
  v[ST_SHADE_DE] = cnt.de_calls;
  v[ST_SHADE_ITERS] = cnt.iterations;
  flush_stats(stats, v);
}

// A distance estimate of the surface shaders at a hit's point plus an offset
// (de_at), as a resumable state.  Deep: an FP32 estimate whose detail is below
// FP32 resolution at its point runs whole in FP64 (calc_distance_p64).
template <class T, int F, bool Deep, int P, int IP>
struct HitDE {
  static constexpr bool kDeep = Deep && sizeof(T) < 8;
  static constexpr bool kWide = kDeep || (formula_march64(F) && sizeof(T) < 8);
  static constexpr bool kAlg = sizeof(T) < 8;
  struct None {};
  DECall<T> c;
  std::conditional_t<kWide, DECall<double>, None> c64;
  bool in64 = false;

  // the estimate in FP64 (trig_DE and the kaleidoscopic IFS have no early end)
  __device__ __forceinline__ bool begin64(const FractalK<double> &fd, V3<double> p, double detail, int N, int minN,
                                          bool normalMode, DEInfo &info) {
    in64 = true;
    double d = 0.0;
    return de_call_begin<double, F, P>(fd, p, detail, N, minN, normalMode, c64, d, info);
  }
  __device__ __forceinline__ double end64(const FractalK<double> &fd, double detail, int N, int minN, bool normalMode,
                                          DEInfo &info) {
    return de_call_end<double, F, P>(fd, c64, detail, N, minN, normalMode, info);
  }

  // true when it ended without iterating (dist and info are then set)
  __device__ __forceinline__ bool begin(const FractalK<double> &fd, const FractalK<T> &f, V3<T> point, V3<double> point64,
                                        V3<T> off, T detail, int N, int minN, bool normalMode, T &dist,
                                        DEInfo &info) {
    if constexpr (kDeep) {
      const V3<double> p = point64 + cvt<double>(off);
      const V3<float> pf = cvt<float>(p);
      const float cmax = length(pf) * (f.julia_mode ? 0.0f : (f.constant_factor > 1.0f ? f.constant_factor : 1.0f));
      const float zc = f.julia_mode ? length(ld3(f.julia)) : cmax;
      in64 = (double)detail < kMixedSwitch * (double)(length(pf) > zc ? length(pf) : zc);
      if (in64) {
        double d = 0.0;
        const bool e = de_call_begin<double, F, P>(fd, p, (double)detail, N, minN, normalMode, c64, d, info);
        dist = (T)d;
        return e;
      }
      return de_call_begin<T, F, P, kAlg, IP>(f, pf, detail, N, minN, normalMode, c, dist, info);
    } else {
      return de_call_begin<T, F, P, kAlg, IP>(f, point + off, detail, N, minN, normalMode, c, dist, info);
    }
  }
  __device__ __forceinline__ bool step(const FractalK<double> &fd, const FractalK<T> &f, int N) {
    if constexpr (kWide) {
      if (in64) return de_call_step<double, F, P>(fd, c64, N);
    }
    return de_call_step<T, F, P, kAlg, IP>(f, c, N);
  }
  __device__ __forceinline__ T end(const FractalK<double> &fd, const FractalK<T> &f, T detail, int N, int minN,
                                   bool normalMode, DEInfo &info) {
    if constexpr (kDeep) {
      if (in64) return (T)de_call_end<double, F, P>(fd, c64, (double)detail, N, minN, normalMode, info);
    }
    return de_call_end<T, F, P, kAlg, IP>(f, c, detail, N, minN, normalMode, info);
  }
};

// The step of the normal's stencil.
template <class T>
__device__ __forceinline__ T stencil_size(const DevScene &sc, const ShaderIn<T> &in) {
  const ShadeK<T> &k = sc.shade<T>();
  if (sc.interior) return in.dist_thresh * k.quality * T(0.2) * k.smoothness;
  return in.delta * k.smoothness;
}

// Surface shading of the hits (ObjectShader's estimates) as three kinds of
// items that depend on the hit's march alone and run side by side: the shadow
// ray (MainShadow, chained estimates), the normal's four estimates (one item
// each; slowShading's stencil has a kernel of its own) and the colouring orbit.  A wave
// works through the shadow rays, then the normals, then the colours; waves
// whose lanes still follow long rays leave the rest of the queues to others.
// One lane per hit instead ran them one after the other at 20-27% active
// lanes and 11-13% VALU busy, and the deep-zoom variant at one wave per SIMD
// (256 + 107 registers).  hit_lit forms the shade from the results: estimates
// in sb.base and sb.spec[0], the shadow factor in sb.spec[1], the detail size
// MainShadow leaves in sb.fast_ao.
enum : int { HIT_SHADOW = 1, HIT_NORMAL = 2, HIT_COLOUR = 4 };
template <class T, int F, bool Deep, int P>
struct HitPolicy {
  static constexpr bool trig64 = (sizeof(T) == 8 && F == 2) || F == 1;
  static constexpr int iters = trig64 ? 2 : 4;
  // waves per SIMD asked of the compiler
  static constexpr int waves = P == kOptions ? 1 : trig64 || (Deep && F == 2) ? 2 : sizeof(T) == 8 || Deep ? 4 : 6;
};

template <class T, int F, bool Deep, int P, int IP>
__global__ void __launch_bounds__(kBlock, (HitPolicy<T, F, Deep, P>::waves))
    k_hits(const DevScene *__restrict__ scp, BandBufs b, SurfBufs<T> sb, int kinds, unsigned long long *stats) {
  const DevScene &sc = *scp;
  constexpr bool kLocal = local_scene(F, P);
  const FractalK<T> f_local = kLocal ? sc.frac<T>() : FractalK<T>{};
  const FractalK<T> &f = kLocal ? f_local : sc.frac<T>();
  constexpr bool kLocal64 = kLocal && (Deep || F == 1) && sizeof(T) < 8;
  const FractalK<double> fd_local = kLocal64 ? sc.fd : FractalK<double>{};
  const FractalK<double> &fd = kLocal64 ? fd_local : sc.fd;
  const ShadeK<T> &k = sc.shade<T>();
  constexpr int kIters = HitPolicy<T, F, Deep, P>::iters;
  const long long n_hits = (long long)b.counters[CNT_HITS];
  const long long n = sb.n;
  const int lane = __lane_id();
  LaneCount cnt = {0, 0};

  if ((kinds & HIT_SHADOW) && sc.shadow) {
    const V3<T> light = v3<T>(k.light[0], k.light[1], k.light[2]);
    const T DE_factor = sc.shadow_fx ? T(1) : k.DE_factor;
    const int N = sc.N, minN = sc.minN, soft = sc.bsoft, fx = sc.shadow_fx, penetrating = sc.penetrating;
    const int iter_fog = sc.iter_fog;
    const T soft_range = k.soft_range;
    const int lanes = item_lanes(n_hits);
    WaveQueue<> queue(&b.counters[CNT_SHADOWQ], n_hits, lanes);
    int state = lane < lanes ? MS_NEED : MS_EXHAUSTED;
    long long tid = 0;
    V3<T> point = v3<T>(0, 0, 0);
    V3<double> point64 = v3<double>(0, 0, 0);
    T i = 0, factor = 0, hit_thr = 0, thr = 0, dist = 0, shadowTemp = 1, maxSoft = 0;
    int guard = 0, early_it = 0;
    bool early = false;
    HitDE<T, F, Deep, P, IP> call;
    auto finish = [&]() __attribute__((always_inline)) {
      sb.spec[n + tid] = soft ? (T(1) - maxSoft) : shadowTemp;
      sb.fast_ao[tid] = thr;  // the detail size MainShadow leaves, for the AO
      state = MS_NEED;
    };
    // the estimate at distance i, or the ray's end
    auto next = [&]() __attribute__((always_inline)) {
      if (!(i < factor && guard < kMaxShadeSteps)) {
        finish();
        return;
      }
      const float dist_thresh = fx ? fx_thresh<T>(sc, point + light * i) : (float)hit_thr;
      thr = (T)dist_thresh;
      DEInfo info;
      early = call.begin(fd, f, point, point64, light * i, thr, N, minN, false, dist, info);
      state = early ? MS_DONE : MS_ITER;
      if (early) early_it = info.iters;
    };
    lane_loop<kIters>(
        state,
        [&](int rank, int n_need) {
          const long long mine = queue.take(b, rank, n_need);
          if (state != MS_NEED) return;
          if (mine < 0) {
            state = MS_EXHAUSTED;
            return;
          }
          tid = mine;
          ShaderIn<T> in;
          load_hit(sc, b, b.hit_list[tid], in);
          point = in.point;
          point64 = in.point64;
          hit_thr = in.dist_thresh;
          factor = in.delta / k.resolution;
          if (!penetrating) factor = k.view_distance_max;
          dist = hit_thr;
          thr = hit_thr;
          i = hit_thr;
          if (sc.interior) i = hit_thr * DE_factor;
          shadowTemp = 1;
          maxSoft = 0;
          guard = 0;
          next();
        },
        [&]() { return call.step(fd, f, N); },
        [&]() {
          int iters = early_it;
          cnt.de_calls += 1;
          if (!early) {
            DEInfo info;
            dist = call.end(fd, f, thr, N, minN, false, info);
            iters = info.iters;
            cnt.iterations += (uint32_t)info.work;
          }
          if (soft) {
            T angle = (dist - thr) / i;
            if (angle < 0) angle = 0;
            if (dist < thr) angle = 0;
            T softShadow = (T(1) - angle / soft_range);
            if (penetrating) softShadow *= (factor - i) / factor;
            if (softShadow < 0) softShadow = 0;
            if (softShadow > maxSoft) maxSoft = softShadow;
          }
          if (iter_fog) shadowTemp -= fog_opacity<T>(sc, dist * DE_factor, iters) * (factor - i) / factor;
          if (dist < thr || shadowTemp < T(0)) {
            shadowTemp -= (factor - i) / factor;
            if (!penetrating) shadowTemp = 0;
            if (shadowTemp < T(0)) shadowTemp = 0;
            finish();
            return;
          }
          i += dist * DE_factor;
          guard++;
          next();
        });
  }

  if (kinds & HIT_NORMAL) {
    // differences of FP32 estimates a stencil step apart keep few digits
    constexpr bool kEst64 = formula_march64(F) && sizeof(T) < 8;
    const int N5 = sc.N * 5;
    const long long n_items = 4 * n_hits;
    const int lanes = item_lanes(n_items);
    WaveQueue<> queue(&b.counters[CNT_NORMALQ], n_items, lanes);
    int state = lane < lanes ? MS_NEED : MS_EXHAUSTED;
    long long item = 0;
    T detail = 0, dist = 0;
    bool early = false;
    HitDE<T, F, Deep, P, IP> call;
    lane_loop<kIters>(
        state,
        [&](int rank, int n_need) {
          const long long mine = queue.take(b, rank, n_need);
          if (state != MS_NEED) return;
          if (mine < 0) {
            state = MS_EXHAUSTED;
            return;
          }
          item = mine;
          ShaderIn<T> in;
          load_hit(sc, b, b.hit_list[item >> 2], in);
          detail = in.detail;
          const T delta = stencil_size<T>(sc, in);
          const int j = (int)(item & 3);
          DEInfo info;
          if constexpr (kEst64) {
            const double d = (double)delta;
            call.begin64(fd, in.point64 + v3<double>(j == 1 ? d : 0.0, j == 2 ? d : 0.0, j == 3 ? d : 0.0),
                         (double)detail, N5, 0, true, info);
            state = MS_ITER;
          } else {
            const V3<T> off = v3<T>(j == 1 ? delta : T(0), j == 2 ? delta : T(0), j == 3 ? delta : T(0));
            early = call.begin(fd, f, in.point, in.point64, off, detail, N5, 0, true, dist, info);
            state = early ? MS_DONE : MS_ITER;
          }
        },
        [&]() { return call.step(fd, f, N5); },
        [&]() {
          cnt.de_calls += 1;
          state = MS_NEED;
          const long long j = item & 3, tid = item >> 2;
          DEInfo info;
          if constexpr (kEst64) {
            sb.est[j][tid] = call.end64(fd, (double)detail, N5, 0, true, info);
            cnt.iterations += (uint32_t)info.work;
          } else {
            if (!early) {
              dist = call.end(fd, f, detail, N5, 0, true, info);
              cnt.iterations += (uint32_t)info.work;
            }
            if (j < 3) sb.base[j * n + tid] = dist;
            else sb.spec[tid] = dist;
          }
        });
  }

  if (kinds & HIT_COLOUR) {
    // whole orbits: their lengths differ little between neighbouring hits
    const int lanes = item_lanes(n_hits);
    WaveQueue<> queue(&b.counters[CNT_COLOURQ], n_hits, lanes);
    for (;;) {
      const long long tid = queue.take(b, lane < lanes ? lane : 64, lanes);
      if (!__ballot(tid >= 0)) break;
      if (tid < 0) continue;
      const int r = b.hit_list[tid];
      ShaderIn<T> in;
      load_hit(sc, b, r, in);
      if (!sc.shadow) sb.fast_ao[tid] = in.detail;
      else if (Deep && sc.shadow_fx) in.detail = sb.fast_ao[tid];
      else in.detail = (T)(float)in.detail;
      put_colour(b, sb, r, tid, surface_colour<T, Deep, formula_march64(F), F, P>(sc, in, cnt));
    }
  }
  poll_before_ao(sc, b);
  unsigned long long v[ST_COUNT] = {0};
  v[ST_SHADE_DE] = cnt.de_calls;
  v[ST_SHADE_ITERS] = cnt.iterations;
  flush_stats(stats, v);
}

// CalculateNormals with slowShading (src/shaders.cpp:720-757): the estimates of
// an 11^3 stencil about the hit, each weighting its offset, summed in the
// reference's order; the sum in sb.base.  A wave per hit and a lane per
// estimate, added up lane by lane.  As a chain of estimates on one lane of
// k_hits a 120x90 FP64 bulb's frame took 14.4 ms, with this 1.4.
template <class T, int F, bool Deep, int P, int IP>
__global__ void __launch_bounds__(kBlock, (HitPolicy<T, F, Deep, P>::waves))
    k_slow_normals(const DevScene *__restrict__ scp, BandBufs b, SurfBufs<T> sb, unsigned long long *stats) {
  const DevScene &sc = *scp;
  constexpr bool kLocal = local_scene(F, P);
  const FractalK<T> f_local = kLocal ? sc.frac<T>() : FractalK<T>{};
  const FractalK<T> &f = kLocal ? f_local : sc.frac<T>();
  const FractalK<double> &fd = sc.fd;
  const int N5 = sc.N * 5, minN = sc.minN;
  const long long n_hits = (long long)b.counters[CNT_HITS];
  const long long n = sb.n;
  const int lane = __lane_id();
  // the stencil's coordinates: the reference's loop variable adds 0.2 up to 1
  int side = 0;
  for (double v = -1.0; v <= 1.0; v += 0.2) side++;
  auto coord = [](int k) {
    double v = -1.0;
    for (int i = 0; i < k; i++) v += 0.2;
    return v;
  };
  const int points = side * side * side;
  LaneCount cnt = {0, 0};
  const long long waves = (long long)gridDim.x * (kBlock / 64);
  for (long long tid = (long long)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); tid < n_hits; tid += waves) {
    ShaderIn<T> in;
    load_hit(sc, b, b.hit_list[tid], in);
    const T delta = stencil_size<T>(sc, in);
    V3<T> sum = v3<T>(0, 0, 0);
    for (int first = 0; first < points; first += 64) {
      const int q = first + lane;
      const V3<T> p2 = v3<T>((T)coord(q / (side * side)), (T)coord(q / side % side), (T)coord(q % side));
      T dist = 0;
      if (q < points) {
        HitDE<T, F, Deep, P, IP> call;
        DEInfo info;
        cnt.de_calls += 1;
        if (!call.begin(fd, f, in.point, in.point64, p2 * delta, in.detail, N5, minN, true, dist, info)) {
          while (!call.step(fd, f, N5)) {
          }
          dist = call.end(fd, f, in.detail, N5, minN, true, info);
          cnt.iterations += (uint32_t)info.work;
        }
      }
      for (int l = 0; l < 64 && first + l < points; l++)
        sum = sum + v3<T>(__shfl(p2.x, l), __shfl(p2.y, l), __shfl(p2.z, l)) * __shfl(dist, l);
    }
    if (lane == 0) {
      sb.base[tid] = sum.x;
      sb.base[n + tid] = sum.y;
      sb.base[2 * n + tid] = sum.z;
    }
  }
  unsigned long long v[ST_COUNT] = {0};
  v[ST_SHADE_DE] = cnt.de_calls;
  v[ST_SHADE_ITERS] = cnt.iterations;
  flush_stats(stats, v);
}

// The normal of hit tid from k_hits's estimates (CalculateNormals).
template <class T>
__device__ __forceinline__ V3<T> hit_normal(const DevScene &sc, const SurfBufs<T> &sb, long long tid) {
  const long long n = sb.n;
  V3<T> v;
  if (sb.est[0]) {
    const double s1 = sb.est[0][tid];
    v = v3<T>((T)(sb.est[1][tid] - s1), (T)(sb.est[2][tid] - s1), (T)(sb.est[3][tid] - s1));
    if (v.x == 0 && v.y == 0 && v.z == 0) v.x = 1;
    else v = normalize(v);
    return v;
  }
  const T s1 = sb.base[tid], s2 = sb.base[n + tid], s3 = sb.base[2 * n + tid];
  v = v3<T>(s1, s2, s3);
  if (!sc.slow_shading) {
    const T s4 = sb.spec[tid];
    v = v3<T>(s2 - s1, s3 - s1, s4 - s1);
  }
  if (v.x == 0 && v.y == 0 && v.z == 0) v.x = 1;
  else v = normalize(v);
  return v;
}

// The lit hit tid from k_hits's results.
template <class T>
__device__ __forceinline__ Lit<T> hit_lit(const DevScene &sc, const BandBufs &b, int band_first, const SurfBufs<T> &sb,
                                          int r, long long tid, ShaderIn<T> &in) {
  load_hit(sc, b, r, in);
  in.view = cvt<T>(ray_dir(sc, b, band_first, r));
  in.normal = hit_normal(sc, sb, tid);
  return light_hit<T>(sc, in, sc.shadow ? sb.spec[sb.n + tid] : T(1));
}

// FastAmbientOcclusion2 of hit tid from k_fast_ao's results; delta: the hit's
// threshold.
template <class T>
__device__ __forceinline__ T fast_ao_of(const DevScene &sc, const SurfBufs<T> &sb, long long tid, long long n_hits,
                                        T delta) {
  if (!sb.fast_items) return sb.spec[2 * sb.n + tid];
  const T tune = sc.shade<T>().fast_ao_tune;
  T aoTemp = 0, inv2i = 1;
  for (int i = 1; i <= sb.fast_items; i++) {
    inv2i *= T(0.5);  // 1/pow(2,i), exact
    const T scan = T(i * i) * delta;
    aoTemp += inv2i * (scan - tune * sb.ao[(i - 1) * n_hits + tid]) / delta;
  }
  const T ao = T(1) - T(0.2) * aoTemp;
  return ao < 0 ? T(0) : ao;
}

// For the shaders that read the lit hits before k_compose (aux and fake
// lights, environment mapping): replaces k_hits's and k_fast_ao's results.
template <class T>
__global__ void __launch_bounds__(kBlock) k_hits_end(const DevScene *__restrict__ scp, BandBufs b, int band_first,
                                                     SurfBufs<T> sb) {
  const DevScene &sc = *scp;
  const long long n_hits = (long long)b.counters[CNT_HITS];
  for (long long tid = (long long)blockIdx.x * kBlock + threadIdx.x; tid < n_hits;
       tid += (long long)gridDim.x * kBlock) {
    ShaderIn<T> in;
    const Lit<T> o = hit_lit<T>(sc, b, band_first, sb, b.hit_list[tid], tid, in);
    in.detail = sb.fast_ao[tid];
    if (sc.ao && sc.fast_ao) sb.fast_ao[tid] = fast_ao_of<T>(sc, sb, tid, n_hits, in.dist_thresh);
    put_lit<T>(sc, in, o, tid, sb);
  }
}

// FastAmbientOcclusion2 (src/shaders.cpp:585-605): quality^2 - 1 estimates
// along each hit's normal.  With room for them (sb.fast_items) every estimate
// is an item of its own, kept in sb.ao for fast_ao_of; else a lane follows a
// hit's estimates one after the other and leaves the AO in sb.spec[2].  An
// estimate inside the set runs all N iterations, and a chain of 15 such ones
// was the kernel's whole time: 400x300 trig_DE, FP32, 5470 us at 6% active
// lanes and 10% VALU busy; as items 920 us (1280x720 power-8 bulb with soft
// shadows, FP32_FIXUP, whole frame: 7.8 -> 5.8 ms with k_hits).
template <class T, int F, bool Deep, int P, int IP>
__global__ void __launch_bounds__(kBlock, (HitPolicy<T, F, Deep, P>::waves))
    k_fast_ao(const DevScene *__restrict__ scp, BandBufs b, SurfBufs<T> sb, unsigned long long *stats) {
  const DevScene &sc = *scp;
  constexpr bool kLocal = local_scene(F, P);
  const FractalK<T> f_local = kLocal ? sc.frac<T>() : FractalK<T>{};
  const FractalK<T> &f = kLocal ? f_local : sc.frac<T>();
  constexpr bool kLocal64 = kLocal && (Deep || F == 1) && sizeof(T) < 8;
  const FractalK<double> fd_local = kLocal64 ? sc.fd : FractalK<double>{};
  const FractalK<double> &fd = kLocal64 ? fd_local : sc.fd;
  const ShadeK<T> &k = sc.shade<T>();
  const long long n_hits = (long long)b.counters[CNT_HITS];
  const long long n = sb.n;
  const int lane = __lane_id();
  const int N = sc.N, minN = sc.minN, end = sc.ao_quality * sc.ao_quality;
  const T tune = k.fast_ao_tune;
  LaneCount cnt = {0, 0};
  const int split = sb.fast_items;
  const long long n_items = split ? n_hits * split : n_hits;
  const int lanes = item_lanes(n_items);
  WaveQueue<> queue(&b.counters[CNT_FASTQ], n_items, lanes);
  int state = lane < lanes ? MS_NEED : MS_EXHAUSTED;
  long long tid = 0;
  V3<T> point = v3<T>(0, 0, 0), normal = point;
  V3<double> point64 = v3<double>(0, 0, 0);
  T delta = 0, detail = 0, dist = 0, aoTemp = 0, inv2i = 1, scan = 0;
  int i = 0;
  bool early = false;
  HitDE<T, F, Deep, P, IP> call;
  auto next = [&]() __attribute__((always_inline)) {
    if (!split && i >= end) {
      T ao = T(1) - T(0.2) * aoTemp;
      if (ao < 0) ao = 0;
      sb.spec[2 * n + tid] = ao;
      state = MS_NEED;
      return;
    }
    inv2i *= T(0.5);  // 1/pow(2,i), exact
    scan = T(i * i) * delta;
    DEInfo info;
    early = call.begin(fd, f, point, point64, normal * scan, detail, N, minN, false, dist, info);
    state = early ? MS_DONE : MS_ITER;
  };
  lane_loop<HitPolicy<T, F, Deep, P>::iters>(
      state,
      [&](int rank, int n_need) {
        const long long mine = queue.take(b, rank, n_need);
        if (state != MS_NEED) return;
        if (mine < 0) {
          state = MS_EXHAUSTED;
          return;
        }
        tid = mine;
        i = 1;
        if (split) {  // (at most 2^21 hits of 63 estimates)
          i = 1 + (int)((unsigned)mine / (unsigned)n_hits);
          tid = mine - (i - 1) * n_hits;
        }
        ShaderIn<T> in;
        load_hit(sc, b, b.hit_list[tid], in);
        point = in.point;
        point64 = in.point64;
        normal = hit_normal(sc, sb, tid);
        delta = in.dist_thresh;
        detail = sb.fast_ao[tid];
        aoTemp = 0;
        inv2i = 1;
        next();
      },
      [&]() { return call.step(fd, f, N); },
      [&]() {
        cnt.de_calls += 1;
        if (!early) {
          DEInfo info;
          dist = call.end(fd, f, detail, N, minN, false, info);
          cnt.iterations += (uint32_t)info.work;
        }
        if (split) {
          sb.ao[(i - 1) * n_hits + tid] = dist;
          state = MS_NEED;
          return;
        }
        aoTemp += inv2i * (scan - tune * dist) / delta;
        i++;
        next();
      });
  unsigned long long v[ST_COUNT] = {0};
  v[ST_SHADE_DE] = cnt.de_calls;
  v[ST_SHADE_ITERS] = cnt.iterations;
  flush_stats(stats, v);
}

// AuxLightsShader (src/shaders.cpp:1051-1073) per hit, after k_hits_end: the
// normal and detail size come from its entries in sb.aux, which are
// replaced by the diffuse and specular sums.  A kernel of its own, so the
// surface kernel of scenes without aux lights keeps its registers.
template <class T, int F, bool Deep>
__global__ void __launch_bounds__(kBlock) k_aux(const DevScene *__restrict__ scp, BandBufs b, int band_first,
                                                SurfBufs<T> sb, unsigned long long *stats) {
  const DevScene &sc = *scp;
  const long long n_hits = (long long)b.counters[CNT_HITS];
  const long long n = sb.n;
  LaneCount cnt = {0, 0};
  for (long long tid = (long long)blockIdx.x * kBlock + threadIdx.x; tid < n_hits;
       tid += (long long)gridDim.x * kBlock) {
    const int r = b.hit_list[tid];
    const V3<double> dir = ray_dir(sc, b, band_first, r);
    ShaderIn<T> in;
    load_hit(sc, b, r, in);
    in.view = cvt<T>(dir);
    in.normal = v3<T>(sb.aux[0 * n + tid], sb.aux[1 * n + tid], sb.aux[2 * n + tid]);
    in.detail = sb.aux[3 * n + tid];
    RGBT<T> al, as;
    aux_lights<T, F, Deep>(sc, in, al, as, cnt);
    if constexpr (sizeof(T) == 8) {
      if (sc.fake_lights) {
        // (auxLights + fakeLights) x colour and auxSpecular + fakeSpecular
        // (ObjectShader, src/shaders.cpp:88-108)
        RGBT<T> fl, fs;
        fake_lights<T>(sc, in, fl, fs, cnt);
        al = RGBT<T>{al.R + fl.R, al.G + fl.G, al.B + fl.B};
        as = RGBT<T>{as.R + fs.R, as.G + fs.G, as.B + fs.B};
      }
    }
    sb.aux[0 * n + tid] = al.R;
    sb.aux[1 * n + tid] = al.G;
    sb.aux[2 * n + tid] = al.B;
    sb.aux[3 * n + tid] = as.R;
    sb.aux[4 * n + tid] = as.G;
    sb.aux[5 * n + tid] = as.B;
  }
  unsigned long long v[ST_COUNT] = {0};
  v[ST_SHADE_DE] = cnt.de_calls;
  v[ST_SHADE_ITERS] = cnt.iterations;
  flush_stats(stats, v);
}

// AmbientOcclusion (src/shaders.cpp:607-673) for all (hit, direction) pairs
// of a band.  Each lane holds one AO ray and advances it one formula
// iteration per loop pass: when its distance estimate completes it takes the
// ray's next step, and when the ray ends it writes the ray's intensity and
// takes the next (hit, direction) item.  Items are handed out per wave from
// a global counter in chunks, so every lane of every wave does formula work
// until the band's AO rays run out, whatever the spread of per-ray step and
// iteration counts.
// Items are (hit, direction) pairs in hit-major order.  A wave walks the
// directions of one hit at a time and takes the next hit index from the
// global counter when they run out, so an item needs no division and a lane
// reloads the hit's data only when its hit changes.
//
// A lane is in one of four states: NEED (wants an item), ITER (advancing a
// distance estimate), DONE (estimate complete, AO step pending) or EXHAUSTED.
// Every pass advances the ITER lanes by up to AOPolicy::iters formula
// iterations (an AO distance estimate of the 1080p power-8 bulb takes 3.6 on
// average).  The AO step logic of DONE lanes runs once 1/done_div of the
// wave waits for it, the item hand-out of NEED lanes once 1/need_div does
// (or nothing else can run), so their cost is shared by many lanes instead
// of being paid on almost every pass.  FP32: 2 iterations, 1/3, 1/8 for the
// Mandelbulb, whose iteration is the longest part of a pass, and 6 iterations
// and 1/2 for the folding formulas, whose iterations are short and more per
// estimate (1280x720 Mandelbox, AO quality 4, FP32_MARCH: AO of a band 7.47 ms
// with 2, 6.92 with 4, 6.86 with 6, the frame 18.3 and 17.1 ms; 1001x563 Menger
// 1.33, 1.25 and 1.22 ms, the frame 2.31 and 2.16).  FP64: 1 iteration, 1/6, 1/8
// (best of the sweeps of the trigonometric Mandelbulb, with 2 waves per SIMD;
// the folding formulas take the same, not swept apart).
enum : int { AO_NEED = 0, AO_ITER = 1, AO_DONE = 2, AO_EXHAUSTED = 3 };
// Per element type: formula iterations per pass, and the share of the wave
// (1/div) that must wait in DONE or NEED before their block runs.
#ifndef MBR_AO_ITERS
#define MBR_AO_ITERS 2
#endif
#ifndef MBR_AO_DONE_DIV
#define MBR_AO_DONE_DIV 3
#endif
#ifndef MBR_AO_NEED_DIV
#define MBR_AO_NEED_DIV 8
#endif
#ifndef MBR_AO64_ITERS
#define MBR_AO64_ITERS 1
#endif
#ifndef MBR_AO64_DONE_DIV
#define MBR_AO64_DONE_DIV 6
#endif
#ifndef MBR_AO64_NEED_DIV
#define MBR_AO64_NEED_DIV 8
#endif
template <class T, int F>
struct AOPolicy {
  static constexpr bool f64 = sizeof(T) == 8;
  static constexpr bool fold = F == 7 || F == 8;
  static constexpr int iters = f64 ? MBR_AO64_ITERS : fold ? 6 : MBR_AO_ITERS;
  static constexpr int done_div = f64 ? MBR_AO64_DONE_DIV : fold ? 2 : MBR_AO_DONE_DIV;
  static constexpr int need_div = f64 ? MBR_AO64_NEED_DIV : MBR_AO_NEED_DIV;
};

template <class T, int F, bool Deep, int Plain, int IP = 0>
__device__ __forceinline__ void ao_body(const DevScene *__restrict__ scp, BandBufs b, AODev ao, SurfBufs<T> sb,
                                        unsigned long long *stats) {
  const DevScene &sc = *scp;
  // trig-free integer-power iteration in FP32, and in FP64 for the fixed power
  constexpr bool kAlg = sizeof(T) < 8 || IP != 0;
  const long long n_hits = (long long)b.counters[CNT_HITS];
  constexpr bool kLocal = local_scene(F, Plain);
  const FractalK<T> f_local = kLocal ? sc.frac<T>() : FractalK<T>{};
  const FractalK<T> &f = kLocal ? f_local : sc.frac<T>();
  const ShadeK<T> &k = sc.shade<T>();
  const T *dirs;
  if constexpr (sizeof(T) == 8) dirs = ao.dir_d; else dirs = ao.dir_f;
  const unsigned count = (unsigned)ao.count;
  const int N = sc.N, minN = sc.minN;
  const int lane = __lane_id();
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));

  // The wave works through units, each 1 / 2^part_bits of a hit's directions:
  // whole hits, or parts of at least 16 directions where there are fewer hits
  // than waves.  Wave-uniform cursor: unit wu (-1 none), next direction wd of it.
  const int waves = (int)gridDim.x * (kBlock / 64);
  int part_bits = 0;
  while ((n_hits << (part_bits + 1)) <= waves && (count >> (part_bits + 1)) >= 16) part_bits++;
  const unsigned unit = (count + (1u << part_bits) - 1) >> part_bits;
  WaveQueue<true> queue(&b.counters[CNT_AOQ], n_hits << part_bits, 1, unit < kRunDirs ? (int)(kRunDirs / unit) : 1,
                        kPollHits + part_bits);
  long long wu = -1;
  unsigned wd = unit;
  int state = AO_NEED;
  long long h_cur = -1;  // hit whose data this lane holds
  unsigned long long item = 0;
  V3<T> P = v3<T>(0, 0, 0), dir = P;
  V3<double> P64 = v3<double>(0, 0, 0);
  bool deep = false;  // FP32 path: the hit's detail is below FP32 resolution of its coordinates
  T r = 0, start_dist = 0, end_dist = 1, detail = 0, thr_f = 0;
  T dist = 0;
  int mi = 0, guard = 0;
  bool early = false;  // the estimate ended in begin_de, without iterating
  DECall<T> call;
  LaneCount cnt = {0, 0};

  // start the distance estimate at P + dir * r; DONE when no iteration runs
  auto begin_de = [&]() {
    DEInfo info;
    const V3<T> p = P + dir * r;
    if constexpr (Deep && sizeof(T) < 8) {
      if (deep)
        early = de_call_begin_p64<F>(sc.fd, f, P64 + cvt<double>(dir) * (double)r, detail, N, minN, false, call, dist,
                                     info);
      else
        early = de_call_begin<T, F, Plain, kAlg, IP>(f, p, detail, N, minN, false, call, dist, info);
    } else {
      early = de_call_begin<T, F, Plain, kAlg, IP>(f, p, detail, N, minN, false, call, dist, info);
    }
    state = early ? AO_DONE : AO_ITER;
    if (early) mi = info.max_iter;
  };

  for (;;) {
    const unsigned long long m_need = __ballot(state == AO_NEED);
    const unsigned long long m_iter = __ballot(state == AO_ITER);
    const unsigned long long m_done = __ballot(state == AO_DONE);
    if (!(m_need | m_iter | m_done)) break;
    const int n_need = __popcll(m_need), n_iter = __popcll(m_iter), n_done = __popcll(m_done);

    if (n_need && (AOPolicy<T, F>::need_div * n_need >= n_need + n_iter + n_done || n_iter + n_done == 0)) {
      // hand out the next items to the lanes that need one, in lane order
      const unsigned n = (unsigned)n_need;
      const unsigned off = (unsigned)__popcll(m_need & lt_mask);
      const unsigned avail = unit - wd;
      long long u = wu;
      unsigned d = wd + off;
      if (n > avail) {
        // new units for the lanes beyond this one's remaining directions
        const unsigned extra = n - avail;
        const unsigned more = (extra + unit - 1) / unit;
        const bool beyond_unit = off >= avail;
        const unsigned j = beyond_unit ? off - avail : 0u;
        const unsigned q = unit >= 64 ? 0u : j / unit;  // several units only when they are small
        const long long got = queue.take(b, (int)q, (int)more);
        if (beyond_unit) {
          // cancelled: no further hits (their AO intensities stay unwritten)
          u = queue.stopped ? -1 : got;
          d = j - q * unit;
        }
        // the last lane that takes one holds the last unit
        wu = __shfl(u, 63 - __builtin_clzll(m_need));
        wd = extra - (more - 1) * unit;
      } else {
        wd += n;
      }
      d += (unsigned)(u & ((1 << part_bits) - 1)) * unit;
      const long long h = u >> part_bits;
      if (state == AO_NEED) {
        if (u < 0) {
          state = AO_EXHAUSTED;
        } else if (d < count) {  // (a hit's last part may be shorter)
          if (h != h_cur) {
            h_cur = h;
            ShaderIn<T> in;
            load_hit(sc, b, b.hit_list[h], in);
            P = in.point;
            P64 = in.point64;
            if constexpr (Deep) deep = (double)in.detail < 2.0 * kMixedSwitch * length(P64);
            start_dist = in.delta;
            end_dist = in.delta / k.resolution;
            detail = sb.fast_ao[h];  // the detail size MainShadow left
            thr_f = (T)(float)in.dist_thresh;  // float dist_thresh (src/shaders.cpp:642)
          }
          item = (unsigned long long)h * count + d;
          dir = v3<T>(dirs[4 * d + 0], dirs[4 * d + 1], dirs[4 * d + 2]);
          r = start_dist;
          guard = 0;
          if (r < end_dist) begin_de();
          else sb.ao[item] = T(1);
        }
      }
    }

    if (state == AO_ITER) {
      bool fin = false;
#pragma unroll
      for (int k = 0; k < AOPolicy<T, F>::iters && !fin; k++)
        fin = de_call_step<T, F, Plain, kAlg, IP>(f, call, N);
      if (fin) state = AO_DONE;
    }

    const unsigned long long m_done2 = __ballot(state == AO_DONE);
    const unsigned long long m_iter2 = __ballot(state == AO_ITER);
    const int n_done2 = __popcll(m_done2), n_iter2 = __popcll(m_iter2);
    if (n_done2 && (AOPolicy<T, F>::done_div * n_done2 >= n_done2 + n_iter2 || n_iter2 == 0) && state == AO_DONE) {
      cnt.de_calls += 1;
      if (!early) {
        DEInfo info;
        dist = de_call_end<T, F, Plain, kAlg, IP>(f, call, detail, N, minN, false, info);
        mi = info.max_iter;
        cnt.iterations += (uint32_t)info.work;
      }
      // one step of the AO ray (src/shaders.cpp:625-662)
      if (dist < thr_f || mi) {
        T shadowTemp = T(1) - (end_dist - r) / end_dist;
        if (shadowTemp < T(0)) shadowTemp = 0;
        sb.ao[item] = shadowTemp;
        state = AO_NEED;
      } else {
        r += dist * T(2);
        guard++;
        if (!(r < end_dist) || guard >= kMaxShadeSteps) {
          sb.ao[item] = T(1);
          state = AO_NEED;
        } else {
          begin_de();
        }
      }
    }
  }
  unsigned long long v[ST_COUNT] = {0};
  v[ST_SHADE_DE] = cnt.de_calls;
  v[ST_SHADE_ITERS] = cnt.iterations;
  v[ST_AO_DE] = cnt.de_calls;
  v[ST_AO_ITERS] = cnt.iterations;
  flush_stats(stats, v);
}

template <class T, int F, bool Deep, int Plain, int IP = 0>
__global__ void __launch_bounds__(kBlock) k_ao(const DevScene *__restrict__ scp, BandBufs b, AODev ao,
                                               SurfBufs<T> sb, unsigned long long *stats) {
  ao_body<T, F, Deep, Plain, IP>(scp, b, ao, sb, stats);
}

// The FP32 plain variant (the benchmarked AO pass) held to 6 waves per SIMD.
template <class T, int F, int Plain, int IP>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6, 8)))
    k_ao_f32_plain(const DevScene *__restrict__ scp, BandBufs b, AODev ao, SurfBufs<T> sb,
                   unsigned long long *stats) {
  ao_body<T, F, false, Plain, IP>(scp, b, ao, sb, stats);
}

// ended: sb.base, sb.spec and sb.fast_ao hold lit hits (k_hits_end, the
// generic surface kernel); else k_hits's results.
//
// A wave composes a run of hits, one per lane; with AmbientOcclusion it first
// sums the AO intensities of four of them at a time, read coalesced: lane j
// takes directions j, j + 64, ... in order, then the 64 partial sums are added
// pairwise (a fixed order, so results are reproducible).
template <class T, class RT>
__global__ void __launch_bounds__(kBlock) k_compose(const DevScene *__restrict__ scp, BandBufs b, int band_first,
                                                    AODev ao, SurfBufs<T> sb, int ended) {
  const DevScene &sc = *scp;
  const long long n_hits = (long long)b.counters[CNT_HITS];
  const ShadeK<T> &k = sc.shade<T>();
  const long long n = sb.n;
  const int lane = __lane_id();
  const long long wave0 = ((long long)blockIdx.x * kBlock + threadIdx.x) / 64;
  const long long waves = (long long)gridDim.x * (kBlock / 64);
  const long long per = (n_hits + waves - 1) / waves;
  const int run = per >= 64 ? 64 : per < 1 ? 1 : (int)per;
  const bool slow_ao = sc.ao && !sc.fast_ao;
  for (long long base = wave0 * run; base < n_hits; base += waves * run) {
    const int here = n_hits - base < run ? (int)(n_hits - base) : run;
    RGBT<T> amb = {0, 0, 0};
    if (slow_ao) {
      for (int q = 0; q < here; q += 4) {
        const T *it = sb.ao + (base + q) * ao.count;
        const int m = here - q < 4 ? here - q : 4;
        RGBT<T> a[4] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
        for (int v = lane; v < ao.count; v += 64) {
          const T cR = T(ao.rgb[4 * v + 0]), cG = T(ao.rgb[4 * v + 1]), cB = T(ao.rgb[4 * v + 2]);
#pragma unroll
          for (int u = 0; u < 4; u++) {
            if (u >= m) break;
            const T s = it[(long long)u * ao.count + v];
            a[u].R += s * cR;
            a[u].G += s * cG;
            a[u].B += s * cB;
          }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
#pragma unroll
          for (int off = 32; off >= 1; off >>= 1) {
            a[u].R += __shfl_xor(a[u].R, off);
            a[u].G += __shfl_xor(a[u].G, off);
            a[u].B += __shfl_xor(a[u].B, off);
          }
          if (lane == q + u) amb = a[u];
        }
      }
      const T den = T(ao.count) * T(256);
      amb.R /= den;
      amb.G /= den;
      amb.B /= den;
    }
    if (lane >= here) continue;
    const long long tid = base + lane;
    const int r = b.hit_list[tid];
    Lit<T> lit;
    if (ended) {
      for (int c = 0; c < 3; c++) {
        lit.base[c] = sb.base[c * n + tid];
        lit.spec[c] = sb.spec[c * n + tid];
      }
    } else {
      ShaderIn<T> in;
      lit = hit_lit<T>(sc, b, band_first, sb, r, tid, in);
    }
    if (sc.ao && sc.fast_ao) {
      const T a = ended ? sb.fast_ao[tid] : fast_ao_of<T>(sc, sb, tid, n_hits, (T)b.thr[r]);
      amb = RGBT<T>{a, a, a};
    }
    const T cR = sb.col[0 * n + tid], cG = sb.col[1 * n + tid], cB = sb.col[2 * n + tid];
    // environment mapping x reflect, times the AO (0 without it)
    RGBT<T> env = {0, 0, 0};
    if (sc.env_map) env = RGBT<T>{sb.aux[6 * n + tid], sb.aux[7 * n + tid], sb.aux[8 * n + tid]};
    if (b.sp_r) {
      // reflections: the object part and the specular part apart
      T oR = env.R * amb.R + (amb.R * k.global_ilum + lit.base[0]) * cR;
      T oG = env.G * amb.G + (amb.G * k.global_ilum + lit.base[1]) * cG;
      T oB = env.B * amb.B + (amb.B * k.global_ilum + lit.base[2]) * cB;
      T sR = lit.spec[0], sG = lit.spec[1], sB = lit.spec[2];
      if (sc.n_lights > 0 || sc.fake_lights) {
        oR += sb.aux[0 * n + tid] * cR;
        oG += sb.aux[1 * n + tid] * cG;
        oB += sb.aux[2 * n + tid] * cB;
        sR = sb.aux[3 * n + tid] + sR;
        sG = sb.aux[4 * n + tid] + sG;
        sB = sb.aux[5 * n + tid] + sB;
      }
      ((RT *)b.sh_r)[r] = (RT)oR;
      ((RT *)b.sh_g)[r] = (RT)oG;
      ((RT *)b.sh_b)[r] = (RT)oB;
      ((RT *)b.sp_r)[r] = (RT)sR;
      ((RT *)b.sp_g)[r] = (RT)sG;
      ((RT *)b.sp_b)[r] = (RT)sB;
    } else if (sc.n_lights > 0 || sc.fake_lights) {
      // (ambient + main light) x colour + aux x colour, then aux specular
      // + main specular (ObjectShader, src/shaders.cpp:96-108)
      ((RT *)b.sh_r)[r] = (RT)(((env.R * amb.R + (amb.R * k.global_ilum + lit.base[0]) * cR) +
                                sb.aux[0 * n + tid] * cR) +
                               (sb.aux[3 * n + tid] + lit.spec[0]));
      ((RT *)b.sh_g)[r] = (RT)(((env.G * amb.G + (amb.G * k.global_ilum + lit.base[1]) * cG) +
                                sb.aux[1 * n + tid] * cG) +
                               (sb.aux[4 * n + tid] + lit.spec[1]));
      ((RT *)b.sh_b)[r] = (RT)(((env.B * amb.B + (amb.B * k.global_ilum + lit.base[2]) * cB) +
                                sb.aux[2 * n + tid] * cB) +
                               (sb.aux[5 * n + tid] + lit.spec[2]));
    } else {
      ((RT *)b.sh_r)[r] = (RT)((env.R * amb.R + (amb.R * k.global_ilum + lit.base[0]) * cR) + lit.spec[0]);
      ((RT *)b.sh_g)[r] = (RT)((env.G * amb.G + (amb.G * k.global_ilum + lit.base[1]) * cG) + lit.spec[1]);
      ((RT *)b.sh_b)[r] = (RT)((env.B * amb.B + (amb.B * k.global_ilum + lit.base[2]) * cB) + lit.spec[2]);
    }
  }
}

// The stages of VolumetricShader that run distance estimates, at a step
// group's point: the volumetric lights (src/shaders.cpp:314-341; stage 0)
// and the iteration fog (:385-465; stage 1), whose record's iteration count
// sets the opacity and the fog colour and whose group is lit by the main
// light and the enabled aux slots through their shadows, plus AO.  `pin` is
// the shader input of the ray's hit, moved to each group's point and
// threshold; b and r name the ray's step records.
template <class T, int F>
struct FxStages {
  const DevScene &sc;
  const BandBufs &b;
  int r;
  ShaderIn<T> &pin;
  LaneCount &cnt;
  const AODev &ao;

  __device__ void iter_fog(int index, T step, VolOut<T> &o, float &totalOpacity) const {
    int L = 0;
    if (index < b.slab) {
      L = b.rec_it[(long long)index * b.cap + r];
    } else {
      const long long dj = b.ovf_off[r];
      const int ch = dj >= 0 ? b.ovf_dir[dj * kDirSlots + (index - b.slab) / kChunk] : -1;
      if (ch >= 0) L = b.ovf_it[(long long)ch * kChunk + (index - b.slab) % kChunk];
    }
    T opacity = iter_opacity<T>(step, T(L), T(sc.N), (T)sc.iter_fog_trim, (T)sc.iter_fog_opacity);
    if (!(opacity > T(0))) return;
    const T trim = (T)sc.iter_fog_trim;
    const T iterFactor = T(2) * (T(L) - trim) / (T(sc.N) - trim);
    T kk = iterFactor;
    if (kk > T(1)) kk = 1;
    if (kk < T(0)) kk = 0;
    T kn = T(1) - kk;
    T fR = T(sc.fog1[0]) * kn + T(sc.fog2[0]) * kk;
    T fG = T(sc.fog1[1]) * kn + T(sc.fog2[1]) * kk;
    T fB = T(sc.fog1[2]) * kn + T(sc.fog2[2]) * kk;
    T k2 = iterFactor - T(1);
    if (k2 < T(0)) k2 = 0;
    if (k2 > T(1)) k2 = 1;
    kn = T(1) - k2;
    fR = fR * kn + T(sc.fog3[0]) * k2;
    fG = fG * kn + T(sc.fog3[1]) * k2;
    fB = fB * kn + T(sc.fog3[2]) * k2;
    const ShadeK<T> &k = sc.shade<T>();
    RGBT<T> nc = {0, 0, 0};
    const T mi = (T)sc.main_light_intensity, dl = k.direct_light;
    if (mi * dl > T(0)) {
      const T sh = main_shadow<T, F>(sc, pin, cnt);
      nc.R += sh * T(sc.main_light_colour[0]) / T(65536) * mi * dl;
      nc.G += sh * T(sc.main_light_colour[1]) / T(65536) * mi * dl;
      nc.B += sh * T(sc.main_light_colour[2]) / T(65536) * mi * dl;
    }
    for (int s4 = 0; s4 < 4; s4++) {
      if (!sc.aux_slot_on[s4]) continue;
      const double *Lt = sc.vol_aux[s4];
      const V3<T> d = v3<T>((T)Lt[0], (T)Lt[1], (T)Lt[2]) - pin.point;
      const T dist = length(d);
      const T d2 = dist * dist;
      const V3<T> lv = normalize(d);
      const T light = aux_shadow<T, F, false>(sc, pin, dist, lv, cnt);
      const T intensity = (T)Lt[3] * T(100);
      nc.R += light * T(Lt[4]) / T(65536) / d2 * intensity;
      nc.G += light * T(Lt[5]) / T(65536) / d2 * intensity;
      nc.B += light * T(Lt[6]) / T(65536) / d2 * intensity;
    }
    if (sc.ao && !sc.fast_ao) {
      AOTable<T> tab;
      if constexpr (sizeof(T) == 8) tab.dir = ao.dir_d; else tab.dir = ao.dir_f;
      tab.rgb = ao.rgb;
      tab.count = ao.count;
      const RGBT<T> a = ambient_occlusion<T, F>(sc, pin, tab, cnt);
      nc.R += a.R * k.global_ilum;
      nc.G += a.G * k.global_ilum;
      nc.B += a.B * k.global_ilum;
    }
    if (opacity > T(1)) opacity = 1;
    o.rgb.R = o.rgb.R * (T(1) - opacity) + nc.R * opacity * fR / T(65536);
    o.rgb.G = o.rgb.G * (T(1) - opacity) + nc.G * opacity * fG / T(65536);
    o.rgb.B = o.rgb.B * (T(1) - opacity) + nc.B * opacity * fB / T(65536);
    totalOpacity = (float)(opacity + (T(1) - opacity) * T(totalOpacity));
    o.alpha = opacity + (T(1) - opacity) * o.alpha;
  }

  __device__ void operator()(int stage, int index, V3<double> p64, T thr, T step, VolOut<T> &o,
                             float &totalOpacity) const {
    pin.point64 = p64;
    pin.point = cvt<T>(p64);
    pin.dist_thresh = thr;
    if (stage == 1) {
      if (sc.iter_fog) iter_fog(index, step, o, totalOpacity);
      return;
    }
    if constexpr (sizeof(T) == 8) {
      if (sc.fake_lights) {
#pragma clang fp contract(off)
        // fake lights' glow (src/shaders.cpp:302-312); 1e-30f is the
        // reference's float literal
        int L = 0;
        T rt = compute<T, MODE_ORBIT_TRAP>(sc.frac<T>(), pin.point, sc.N, &L);
        cnt.de_calls += 1;
        rt = Math<T>::sqrt(T(1) / (rt + T(1.0e-30f)));
        const T e = T(10) / T(sc.fl_visibility_size);
        const T glow = T(1) / (Math<T>::pow(rt, e) * Math<T>::pow(T(10), e) + T(1e-100));
        const T v = T(sc.fl_visibility);
        o.rgb.R += glow * step * v;
        o.rgb.G += glow * step * v;
        o.rgb.B += glow * step * v;
        o.alpha += glow * step * v;
      }
    }
    if (sc.vol_main) {
      const T sh = main_shadow<T, F>(sc, pin, cnt);
      const T I0 = (T)sc.vol_intensity[0];
      o.rgb.R += sh * step * I0 * T(sc.main_light_colour[0]) / T(65536);
      o.rgb.G += sh * step * I0 * T(sc.main_light_colour[1]) / T(65536);
      o.rgb.B += sh * step * I0 * T(sc.main_light_colour[2]) / T(65536);
      o.alpha += (sh + sh + sh) / T(3) * step * I0;
    }
    for (int k = 0; k < 4; k++) {
      if (!sc.vol_aux_on[k]) continue;
      const double *L = sc.vol_aux[k];
      const V3<T> d = v3<T>((T)L[0], (T)L[1], (T)L[2]) - pin.point;
      const T dl = length(d);
      const T d2 = dl * dl;
      const V3<T> lv = normalize(d);
      const T light = aux_shadow<T, F, false>(sc, pin, dl, lv, cnt);
      const T Ik = (T)sc.vol_intensity[k + 1];
      o.rgb.R += light * T(L[4]) / T(65536) * Ik * step / d2;
      o.rgb.G += light * T(L[5]) / T(65536) * Ik * step / d2;
      o.rgb.B += light * T(L[6]) / T(65536) * Ik * step / d2;
      o.alpha += light * Ik * step / d2;
    }
  }
};

// ---------------------------------------------------------------- finish
// One pixel: background or shaded surface, then VolumetricShader over the
// ray's step records.  FX: the volumetric lights' shadow marches run here
// (distance estimates of formula F).
template <class T, class RT, int F, bool FX, bool VIS>
__device__ __forceinline__ void finish_body(const DevScene &sc, const BandBufs &b, int band_first, int r,
                                            const FrameOut &out, LaneCount &cnt, const AODev &ao) {
  const int p = band_first + r;
  const bool found = b.found[r];
  RGBT<T> px;
  T alpha;
  uint8_t cr = 0, cg = 0, cb = 0;
  if (found) {
    px = RGBT<T>{(T)((const RT *)b.sh_r)[r], (T)((const RT *)b.sh_g)[r], (T)((const RT *)b.sh_b)[r]};
    alpha = 1;
    cr = b.col_r[r]; cg = b.col_g[r]; cb = b.col_b[r];
  } else {
    const int x = p % sc.width, y = p / sc.width;
    V3<double> dir;
    view_vector(sc, x, y, dir);
    RGBT<double> bg = background<double>(sc, dir);
    px = RGBT<T>{(T)bg.R, (T)bg.G, (T)bg.B};
    alpha = 0;
  }
  const int n = b.count[r];
  const T depth = (T)b.depth[r];
  VolOut<T> v;
  const RT *st = (const RT *)b.rec_step, *di = (const RT *)b.rec_dist, *th = (const RT *)b.rec_thr;
  const long long cap = b.cap;
  const int slab = b.slab;
  // visible aux lights glow along the ray: its direction and the scan of
  // the last record (the sum of all recorded steps)
  VisRay vray;
  const VisRay *vr = nullptr;
  const bool vis = VIS && sc.n_lights > 0 && sc.sd.aux_visibility > 0;
  if (vis || FX) {
    const int x = p % sc.width, y = p / sc.width;
    view_vector(sc, x, y, vray.dir);
    vray.start = v3<double>(sc.start[0], sc.start[1], sc.start[2]);
    vr = &vray;
  }
  // the volumetric lights of a step group (src/shaders.cpp:314-341), from
  // the shader input of the pixel with the group's point and threshold
  ShaderIn<T> pin;
  if constexpr (FX) {
    load_hit(sc, b, r, pin);
    pin.view = cvt<T>(vray.dir);
  }
  auto fx = [&](int stage, int index, V3<double> p64, T thr, T step, VolOut<T> &o, float &totalOpacity) {
    if constexpr (FX) {
      FxStages<T, F>{sc, b, r, pin, cnt, ao}(stage, index, p64, thr, step, o, totalOpacity);
    } else {
      (void)stage; (void)index; (void)p64; (void)thr; (void)step; (void)o; (void)totalOpacity;
    }
  };
  if (n <= slab) {
    auto rec = [&](int i, T &s, T &d, T &t) {
      const long long o = (long long)i * cap + r;
      s = (T)st[o]; d = (T)di[o]; t = (T)th[o];
    };
    if (vr) {
      double sum = 0.0;
      for (int i = 0; i < n; i++) sum += (double)st[(long long)i * cap + r];
      vray.scan_end = sum;
    }
    v = volumetric<FX || VIS ? 1 : 4>(sc, depth, n, px, alpha, rec, vr, vis, fx);
  } else {
    // records from the slab on sit in the chunks the ray's directory lists
    // (the host renders a band again when a record found the pool full)
    const RT *ost = (const RT *)b.ovf_step, *odi = (const RT *)b.ovf_dist, *oth = (const RT *)b.ovf_thr;
    const long long dj = b.ovf_off[r];
    const int *dir = b.ovf_dir + (dj >= 0 ? dj : 0) * kDirSlots;
    auto rec = [&](int i, T &s, T &d, T &t) {
      const int ch = (i >= slab && dj >= 0) ? dir[(i - slab) / kChunk] : -1;
      if (i < slab) {
        const long long o = (long long)i * cap + r;
        s = (T)st[o]; d = (T)di[o]; t = (T)th[o];
      } else if (ch >= 0) {
        const long long o = (long long)ch * kChunk + (i - slab) % kChunk;
        s = (T)ost[o]; d = (T)odi[o]; t = (T)oth[o];
      } else {
        s = 0; d = 0; t = 0;
      }
    };
    if (vr) {
      double sum = 0.0;
      for (int i = 0; i < n; i++) {
        T s, d, t;
        rec(i, s, d, t);
        sum += (double)s;
      }
      vray.scan_end = sum;
    }
    v = volumetric<FX || VIS ? 1 : 4>(sc, depth, n, px, alpha, rec, vr, vis, fx);
  }
  if (out.rgb[0]) out.rgb[0][p] = (float)v.rgb.R;
  if (out.rgb[1]) out.rgb[1][p] = (float)v.rgb.G;
  if (out.rgb[2]) out.rgb[2][p] = (float)v.rgb.B;
  if (out.z) out.z[p] = found ? (float)b.depth[r] : 1e20f;
  if (out.colour[0]) out.colour[0][p] = cr;
  if (out.colour[1]) out.colour[1][p] = cg;
  if (out.colour[2]) out.colour[2][p] = cb;
  if (out.opacity) out.opacity[p] = x86_d2u16((double)v.opacity * 65535.0);
  if (out.alpha) out.alpha[p] = x86_d2u16((double)v.alpha * 65535.0);
}

// VIS: the variant with the glow of visible aux lights
template <class T, class RT, bool VIS>
__global__ void __launch_bounds__(kBlock) k_finish(const DevScene *__restrict__ scp, BandBufs b, int band_first,
                                                   int band_rays, FrameOut out) {
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r >= band_rays) return;
  LaneCount cnt = {0, 0};
  finish_body<T, RT, 0, false, VIS>(*scp, b, band_first, r, out, cnt, AODev{});
}

// With volumetric lights: a grid-stride loop (the shadow marches make the
// per-pixel cost vary widely), distance-estimate counts into the stats.
template <class T, class RT, int F>
__global__ void __launch_bounds__(kBlock) k_finish_fx(const DevScene *__restrict__ scp, BandBufs b, int band_first,
                                                      int band_rays, FrameOut out, unsigned long long *stats,
                                                      AODev ao) {
  LaneCount cnt = {0, 0};
  for (int r = blockIdx.x * kBlock + threadIdx.x; r < band_rays; r += gridDim.x * kBlock)
    finish_body<T, RT, F, true, true>(*scp, b, band_first, r, out, cnt, ao);
  unsigned long long v[ST_COUNT] = {0};
  v[ST_SHADE_DE] = cnt.de_calls;
  v[ST_SHADE_ITERS] = cnt.iterations;
  flush_stats(stats, v);
}

// ----------------------------------------------------------- reflections
#if MBR_UNIT(5)
__global__ void k_refl_clear(uint8_t *active, int n) {
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r < n) active[r] = 0;
}
#endif

// The mirrored rays of the reflecting hits of `prev` (src/Render3D.cpp:
// 478-498): normal at the hit (CalculateNormals with the hit's threshold as
// detail size), view vector mirrored about it, start one threshold along it.
template <int F>
__global__ void __launch_bounds__(kBlock) k_refl_setup(const DevScene *__restrict__ scp, BandBufs prev, BandBufs next,
                                                       int band_first, unsigned long long *stats) {
  const DevScene &sc = *scp;
  const long long n_hits = (long long)prev.counters[CNT_HITS];
  LaneCount cnt = {0, 0};
  for (long long t = (long long)blockIdx.x * kBlock + threadIdx.x; t < n_hits; t += (long long)gridDim.x * kBlock) {
    const int r = prev.hit_list[t];
    if (sc.refl[prev.object[r] % 7] == 0.0) continue;
    const V3<double> dir = ray_dir(sc, prev, band_first, r);
    ShaderIn<double> in;
    load_hit(sc, prev, r, in);
    in.view = dir;
    const V3<double> n = normals<double, F>(sc, in, cnt);
    const V3<double> d2 = dir - (n * dot(dir, n)) * 2.0;
    const double thr = prev.thr[r];
    const V3<double> o = in.point64 + d2 * thr;
    next.ray_o[3 * (long long)r + 0] = o.x;
    next.ray_o[3 * (long long)r + 1] = o.y;
    next.ray_o[3 * (long long)r + 2] = o.z;
    next.ray_d[3 * (long long)r + 0] = d2.x;
    next.ray_d[3 * (long long)r + 1] = d2.y;
    next.ray_d[3 * (long long)r + 2] = d2.z;
    next.ray_t0[r] = thr;
    next.active[r] = 1;
    next.hand_ray[atomicAdd(&next.counters[CNT_HAND], 1ull)] = r;
  }
  unsigned long long v[ST_COUNT] = {0};
  v[ST_SHADE_DE] = cnt.de_calls;
  v[ST_SHADE_ITERS] = cnt.iterations;
  flush_stats(stats, v);
}

// Per pixel: the levels from the last one reached down to the primary ray
// (src/Render3D.cpp:501-571): each shaded surface (or background) blended
// with the next level's result by its reflection coefficient, then that
// level's VolumetricShader over its own step records.  FX: with volumetric
// lights or iteration fog, each level's VolumetricShader runs their shadow
// marches (formula F) from that level's hit, as the primary ray's does.
template <int F, bool VIS, bool FX>
__global__ void __launch_bounds__(kBlock) k_refl_finish(const DevScene *__restrict__ scp,
                                                        const BandBufs *__restrict__ levels, int n_levels,
                                                        int band_first, int band_rays, FrameOut out, AODev ao,
                                                        unsigned long long *stats) {
  const DevScene &sc = *scp;
  LaneCount cnt = {0, 0};
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r < band_rays) {
  const int p = band_first + r;
  int rayEnd = 0;
  for (int k = 1; k < n_levels; k++) {
    if (!levels[k].active[r]) break;
    rayEnd = k;
  }
  const int maxRay = n_levels - 1;
  RGBT<double> result = {0, 0, 0};
  double opacity0 = 0, alpha0 = 0;
  for (int ray = rayEnd; ray >= 0; ray--) {
    const BandBufs &b = levels[ray];
    const bool found = b.found[r];
    const V3<double> dir = ray_dir(sc, b, band_first, r);
    RGBT<double> obj = {0, 0, 0}, bg = {0, 0, 0}, spec = {0, 0, 0};
    if (found) {
      obj = RGBT<double>{((const double *)b.sh_r)[r], ((const double *)b.sh_g)[r], ((const double *)b.sh_b)[r]};
      spec = RGBT<double>{((const double *)b.sp_r)[r], ((const double *)b.sp_g)[r], ((const double *)b.sp_b)[r]};
    } else {
      bg = background<double>(sc, dir);
    }
    const double reflect = sc.refl[b.object[r] % 7];
    RGBT<double> px;
    if (maxRay > 0 && rayEnd > 0 && ray != rayEnd) {
      px.R = result.R * reflect + (1.0 - reflect) * (obj.R + bg.R) + spec.R;
      px.G = result.G * reflect + (1.0 - reflect) * (obj.G + bg.G) + spec.G;
      px.B = result.B * reflect + (1.0 - reflect) * (obj.B + bg.B) + spec.B;
    } else {
      px.R = obj.R + bg.R + spec.R;
      px.G = obj.G + bg.G + spec.G;
      px.B = obj.B + bg.B + spec.B;
    }
    const double alpha = found ? 1.0 : 0.0;
    const int n = b.count[r];
    const double depth = b.depth[r];
    const double *st = (const double *)b.rec_step, *di = (const double *)b.rec_dist, *th = (const double *)b.rec_thr;
    const double *ost = (const double *)b.ovf_step, *odi = (const double *)b.ovf_dist, *oth = (const double *)b.ovf_thr;
    const long long cap = b.cap;
    const int slab = b.slab;
    const long long dj = b.ovf_off[r];
    auto rec = [&](int i, double &s, double &d, double &t) {
      if (i < slab) {
        const long long o = (long long)i * cap + r;
        s = st[o]; d = di[o]; t = th[o];
        return;
      }
      const int ch = dj >= 0 ? b.ovf_dir[dj * kDirSlots + (i - slab) / kChunk] : -1;
      if (ch >= 0) {
        const long long o = (long long)ch * kChunk + (i - slab) % kChunk;
        s = ost[o]; d = odi[o]; t = oth[o];
      } else {
        s = 0; d = 0; t = 0;
      }
    };
    VisRay vray;
    const VisRay *vr = nullptr;
    const bool vis = VIS && sc.n_lights > 0 && sc.sd.aux_visibility > 0;
    if (vis || FX) {
      vray.dir = dir;
      vray.start = ray == 0 ? v3<double>(sc.start[0], sc.start[1], sc.start[2])
                            : v3<double>(b.ray_o[3 * (long long)r], b.ray_o[3 * (long long)r + 1],
                                         b.ray_o[3 * (long long)r + 2]);
      double sum = 0.0;
      for (int i = 0; i < n; i++) {
        double s_, d_, t_;
        rec(i, s_, d_, t_);
        sum += s_;
      }
      vray.scan_end = sum;
      vr = &vray;
    }
    ShaderIn<double> pin;
    if constexpr (FX) {
      load_hit(sc, b, r, pin);
      pin.view = dir;
    }
    auto fx = [&](int stage, int index, V3<double> p64, double thr, double step, VolOut<double> &o,
                  float &totalOpacity) {
      if constexpr (FX) {
        FxStages<double, F>{sc, b, r, pin, cnt, ao}(stage, index, p64, thr, step, o, totalOpacity);
      } else {
        (void)stage; (void)index; (void)p64; (void)thr; (void)step; (void)o; (void)totalOpacity;
      }
    };
    const VolOut<double> v = volumetric<FX || VIS ? 1 : 4>(sc, depth, n, px, alpha, rec, vr, vis, fx);
    result = v.rgb;
    if (ray == 0) {
      opacity0 = v.opacity;
      alpha0 = v.alpha;
    }
  }
  const BandBufs &b0 = levels[0];
  const bool found0 = b0.found[r];
  if (out.rgb[0]) out.rgb[0][p] = (float)result.R;
  if (out.rgb[1]) out.rgb[1][p] = (float)result.G;
  if (out.rgb[2]) out.rgb[2][p] = (float)result.B;
  if (out.z) out.z[p] = found0 ? (float)b0.depth[r] : 1e20f;
  if (out.colour[0]) out.colour[0][p] = found0 ? b0.col_r[r] : 0;
  if (out.colour[1]) out.colour[1][p] = found0 ? b0.col_g[r] : 0;
  if (out.colour[2]) out.colour[2][p] = found0 ? b0.col_b[r] : 0;
  if (out.opacity) out.opacity[p] = x86_d2u16(opacity0 * 65535.0);
  if (out.alpha) out.alpha[p] = x86_d2u16(alpha0 * 65535.0);
  }
  if constexpr (FX) {
    unsigned long long v[ST_COUNT] = {0};
    v[ST_SHADE_DE] = cnt.de_calls;
    v[ST_SHADE_ITERS] = cnt.iterations;
    flush_stats(stats, v);
  }
}

// ---------------------------------------------------------------- launch
// Calls go(F, Plain, IP) (as integral constants) with the compiled variant of
// a scene: the formula's kernels (0: generic), without the optional terms of
// the distance estimate where the scene has none, and with the Mandelbulb's
// power 8 fixed where the trig-free iteration is wanted (ip8).
template <class Go>
static inline void march_variant(int formula, int plain, bool ip8, Go go) {
  std::integral_constant<int, 0> z;
  std::integral_constant<int, 2> f2;
  std::integral_constant<int, 7> f7;
  std::integral_constant<int, 8> f8;
  std::integral_constant<int, kPlain> yes;
  std::integral_constant<int, kOptions> no;
  std::integral_constant<int, kStandardBox> box;
  // trig_DE and the kaleidoscopic IFS: compiled by themselves their march takes
  // 226 and 122 registers and no scratch memory (trig_DE's FP32 AO spills 10 of
  // its 80), the generic ones (30 formulas, finite differences, whole estimates)
  // 512 and 1.8 KB.  400x300 trig_DE with
  // soft shadows and fast AO, FP32_FIXUP: 15.6 -> 10.4 ms (march 5.5 -> 1.4).
  // The optional terms stay with the generic kernels.
  if (formula_march64(formula) && plain) {
    std::integral_constant<int, 1> f1;
    std::integral_constant<int, 10> f10;
    return formula == 1 ? go(f1, yes, z) : go(f10, yes, z);
  }
  if (formula_generic(formula)) return go(z, no, z);
  if (plain) {
    if (formula == 7) return go(f7, yes, z);
    if (formula == 8) return plain == kStandardBox ? go(f8, box, z) : go(f8, yes, z);
    return ip8 ? go(f2, yes, f8) : go(f2, yes, z);
  }
  if (formula == 7) return go(f7, no, z);
  if (formula == 8) return go(f8, no, z);
  return ip8 ? go(f2, no, f8) : go(f2, no, z);
}

static inline dim3 grid_for(int n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); }

#if MBR_UNIT(5)
hipError_t launch_refl_clear(const BandBufs &next, int band_rays, hipStream_t s) {
  if (band_rays <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_refl_clear, grid_for(band_rays), dim3(kBlock), 0, s, next.active, band_rays);
  return hipGetLastError();
}

hipError_t launch_refl_setup(const DevScene *sc, const BandBufs &prev, const BandBufs &next, int band_first,
                             int formula, int blocks, unsigned long long *stats, hipStream_t s) {
  const dim3 grid((unsigned)std::max(1, blocks));
  if (formula_generic(formula))
    hipLaunchKernelGGL((k_refl_setup<0>), grid, dim3(kBlock), 0, s, sc, prev, next, band_first, stats);
  else if (formula == 7)
    hipLaunchKernelGGL((k_refl_setup<7>), grid, dim3(kBlock), 0, s, sc, prev, next, band_first, stats);
  else if (formula == 8)
    hipLaunchKernelGGL((k_refl_setup<8>), grid, dim3(kBlock), 0, s, sc, prev, next, band_first, stats);
  else
    hipLaunchKernelGGL((k_refl_setup<2>), grid, dim3(kBlock), 0, s, sc, prev, next, band_first, stats);
  return hipGetLastError();
}

hipError_t launch_refl_march(const DevScene *sc, const BandBufs &next, int band_first, int formula, int blocks,
                             unsigned long long *stats, hipStream_t s) {
  if (formula_generic(formula))
    launch_resident<k_march64<double, 0, 0, 0, kRefl>>(blocks, s, sc, next, band_first, 0, stats);
  else if (formula == 7)
    launch_resident<k_march64<double, 7, 0, 0, kRefl>>(blocks, s, sc, next, band_first, 0, stats);
  else if (formula == 8)
    launch_resident<k_march64<double, 8, 0, 0, kRefl>>(blocks, s, sc, next, band_first, 0, stats);
  else
    launch_resident<k_march64<double, 2, 0, 0, kRefl>>(blocks, s, sc, next, band_first, 0, stats);
  return hipGetLastError();
}

hipError_t launch_refl_finish(const DevScene *sc, const BandBufs *levels, int n_levels, int band_first,
                              int band_rays, FrameOut out, int vis, int fx, int formula, AODev ao,
                              unsigned long long *stats, hipStream_t s) {
  if (band_rays <= 0) return hipSuccess;
  const dim3 grid = grid_for(band_rays);
  auto run = [&](auto ftag) {
    constexpr int F = decltype(ftag)::value;
    if (fx)
      hipLaunchKernelGGL((k_refl_finish<F, true, true>), grid, dim3(kBlock), 0, s, sc, levels, n_levels, band_first,
                         band_rays, out, ao, stats);
    else if (vis)
      hipLaunchKernelGGL((k_refl_finish<0, true, false>), grid, dim3(kBlock), 0, s, sc, levels, n_levels,
                         band_first, band_rays, out, ao, stats);
    else
      hipLaunchKernelGGL((k_refl_finish<0, false, false>), grid, dim3(kBlock), 0, s, sc, levels, n_levels,
                         band_first, band_rays, out, ao, stats);
  };
  if (!fx || formula_generic(formula)) run(std::integral_constant<int, 0>{});
  else if (formula == 7) run(std::integral_constant<int, 7>{});
  else if (formula == 8) run(std::integral_constant<int, 8>{});
  else run(std::integral_constant<int, 2>{});
  return hipGetLastError();
}

#endif  // reflections

#if MBR_UNIT(0)
hipError_t launch_march(int precision, const DevScene *sc, const BandBufs &b, int band_first, int band_rays,
                        int formula, int plain, int persist_blocks, unsigned long long *stats, hipStream_t s,
                        bool ip8) {
  if (band_rays <= 0) return hipSuccess;
  // generic formulas: FP64, or the FP64 march of FP32_FIXUP (FP32 records)
  if (formula_generic(formula) && precision > 1) return hipErrorInvalidValue;
  if (precision == 2) {
    auto go = [&](auto f_tag, auto plain_tag, auto ip_tag) {
      constexpr int F = decltype(f_tag)::value;
      if constexpr (F != 0 && !formula_march64(F))
        launch_resident<k_march<F, decltype(plain_tag)::value, decltype(ip_tag)::value>>(persist_blocks, s, sc, b,
                                                                                         band_first, band_rays, stats);
    };
    march_variant(formula, plain, ip8, go);
    return hipGetLastError();
  }
  auto run = [&](auto rtag) {
    using RT = decltype(rtag);
    auto go = [&](auto f_tag, auto plain_tag, auto ip_tag) {
      constexpr int F = decltype(f_tag)::value, Pl = decltype(plain_tag)::value, IP = decltype(ip_tag)::value;
      launch_resident<k_march64<RT, F, Pl, IP, kRays>>(persist_blocks, s, sc, b, band_first, band_rays, stats);
    };
    march_variant(formula, plain, ip8, go);
  };
  if (precision == 0) run(double{});
  else run(float{});
  return hipGetLastError();
}
#endif  // march

#if MBR_UNIT(1)
hipError_t launch_march_fix(const DevScene *sc, const BandBufs &b, int band_first, int formula, int plain,
                            int persist_blocks, unsigned long long *stats, hipStream_t s, bool ip8) {
  if (formula_generic(formula)) return hipErrorInvalidValue;
  auto hand = [&](auto f_tag, auto plain_tag, auto ip_tag) {
    constexpr int F = decltype(f_tag)::value, IP = decltype(ip_tag)::value;
    constexpr int Pl = decltype(plain_tag)::value;
    if constexpr (F != 0 && !formula_march64(F)) {
      launch_resident<k_march64<float, F, Pl, IP, kHand>>(persist_blocks, s, sc, b, band_first, 0, stats);
      launch_resident<k_march64<float, F, Pl, IP, kRedo>>(persist_blocks, s, sc, b, band_first, 0, stats);
    }
  };
  march_variant(formula, plain, ip8, hand);
  return hipGetLastError();
}
#endif  // continuation

#if MBR_UNIT(4)
// Clears a band's counters; a render cancelled by now starts its band stopped.
__global__ void k_band_reset(BandBufs b) {
  const int i = (int)threadIdx.x;
  if (i >= CNT_COUNT) return;
  const bool stop = (i == CNT_RAYQ || i == CNT_AOQ) && b.cancel && *b.cancel != 0;
  b.counters[i] = stop ? kStopBit : 0;
}

hipError_t launch_band_reset(const BandBufs &b, hipStream_t s) {
  hipLaunchKernelGGL(k_band_reset, dim3(1), dim3(64), 0, s, b);
  return hipGetLastError();
}

__global__ void k_zero(unsigned long long *p, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0;
}

hipError_t launch_zero(unsigned long long *p, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_zero, dim3(1), dim3(64), 0, s, p, n);
  return hipGetLastError();
}

#endif  // resets

// The shading launches of one element type (T: the path's precision).
template <class T>
hipError_t shade_run(const DevScene *sc, const BandBufs &b, int band_first, AODev ao, ShadeBufs sbuf,
                     int persist_blocks, unsigned long long *stats, hipStream_t s, hipEvent_t ev_ao0,
                     hipEvent_t ev_ao1);

#if MBR_UNIT(2) || MBR_UNIT(3)
template <class T>
hipError_t shade_run(const DevScene *sc, const BandBufs &b, int band_first, AODev ao, ShadeBufs sbuf,
                     int persist_blocks, unsigned long long *stats, hipStream_t s, hipEvent_t ev_ao0,
                     hipEvent_t ev_ao1) {
  const int formula = sbuf.formula;
  // persistent grids: enough workgroups to fill every CU several times; the
  // kernels loop over the band's hits
  const dim3 grid((unsigned)std::max(1, persist_blocks));
  SurfBufs<T> sb;
  sb.base = (T *)sbuf.base;
  sb.spec = (T *)sbuf.spec;
  sb.col = (T *)sbuf.col;
  sb.fast_ao = (T *)sbuf.fast_ao;
  sb.ao = (T *)sbuf.ao;
  sb.aux = (T *)sbuf.aux;
  sb.n = sbuf.n;
  sb.fast_items = sbuf.fast_items;
  const bool generic = formula_generic(formula);
  // generic formulas with kernels of their own
  const bool own = generic && sbuf.plain && formula_march64(formula);
  const bool est64 = own && sizeof(T) < 8 && !sbuf.slow_normals;
  double *const planes[4] = {b.hand_scan, b.hand_step, b.hand_drift, b.hand_dist};
  for (int i = 0; i < 4; i++) sb.est[i] = est64 ? planes[i] : nullptr;
  // deep-zoom variants only for FP32 shading of scenes that need them
  const bool deep = sbuf.deep && sizeof(T) < 8 && !generic;
  // the variants of the surface kernels; FP64 shades with the reference's
  // trigonometric iteration
  auto variants = [&](auto go) {
    march_variant(formula, sbuf.plain, sbuf.ip8 && sizeof(T) < 8, [&](auto f_tag, auto plain_tag, auto ip_tag) {
      if constexpr (decltype(f_tag)::value != 0) {
        constexpr int IP = sizeof(T) < 8 ? decltype(ip_tag)::value : 0;
        std::integral_constant<int, IP> ip;
        if constexpr (sizeof(T) < 8 && !formula_march64(decltype(f_tag)::value)) {
          if (deep) return go(std::true_type{}, f_tag, plain_tag, ip);
        }
        go(std::false_type{}, f_tag, plain_tag, ip);
      }
    });
  };
  auto hits = [&](int kinds) {
    variants([&](auto d, auto f, auto pl, auto ip) {
      constexpr int F = decltype(f)::value, Pl = decltype(pl)::value, IP = decltype(ip)::value;
      if ((kinds & HIT_NORMAL) && sbuf.slow_normals) {
        launch_resident<k_slow_normals<T, F, decltype(d)::value, Pl, IP>>(persist_blocks, s, sc, b, sb, stats);
        kinds &= ~HIT_NORMAL;
      }
      // deep zooms: a quarter of the workgroups (2 per CU), which keep the FP64
      // units busy and leave room for the other stream's march (4K Mandelbox
      // 78.4 ms with as many as fit, 76.4 with 4 per CU, 75.6 with 2; 1280x720
      // 14.1, 13.5 with 3 and 13.0 with 2; 640x360 on one stream 6.2 and 6.0)
      const int blocks = decltype(d)::value ? persist_blocks / 4 : persist_blocks;
      launch_resident<k_hits<T, F, decltype(d)::value, Pl, IP>>(blocks, s, sc, b, sb, kinds, stats);
    });
  };
  // plain scenes take a variant without the optional terms' branches (and the
  // scene constants they keep live); FP32 deep-zoom scenes the one that starts
  // estimates in FP64
  auto aok = [&](auto deep_tag, auto f_tag, auto plain_tag, auto ip_tag) {
    constexpr bool D = decltype(deep_tag)::value;
    constexpr int F = decltype(f_tag)::value, Pl = decltype(plain_tag)::value, IP = decltype(ip_tag)::value;
    if constexpr (!D && Pl && std::is_same<T, float>::value)
      launch_resident<k_ao_f32_plain<T, F, Pl, IP>>(persist_blocks, s, sc, b, ao, sb, stats);
    else if constexpr (Pl)
      launch_resident<k_ao<T, F, D, Pl, IP>>(persist_blocks, s, sc, b, ao, sb, stats);
    else
      launch_resident<k_ao<T, F, D, Pl>>(persist_blocks, s, sc, b, ao, sb, stats);
  };
  int ended = 0;
  if (generic && !own) {
    hipLaunchKernelGGL((k_surface_generic<T>), grid, dim3(kBlock), 0, s, sc, b, band_first, sb, stats);
    ended = 1;
  } else {
    // the colour of a deep hit under shadow_fx depends on the detail size its
    // shadow ray left
    if (deep && sbuf.shadow_fx) {
      hits(HIT_SHADOW | HIT_NORMAL);
      hits(HIT_COLOUR);
    } else {
      hits(HIT_SHADOW | HIT_NORMAL | HIT_COLOUR);
    }
    if (sbuf.fast_ao_on)
      variants([&](auto d, auto f, auto pl, auto ip) {
        constexpr int F = decltype(f)::value, Pl = decltype(pl)::value, IP = decltype(ip)::value;
        launch_resident<k_fast_ao<T, F, decltype(d)::value, Pl, IP>>(persist_blocks, s, sc, b, sb, stats);
      });
    if (sbuf.lights || sbuf.env) {
      hipLaunchKernelGGL((k_hits_end<T>), grid, dim3(kBlock), 0, s, sc, b, band_first, sb);
      ended = 1;
    }
  }
  if (sbuf.lights) {
    if (generic) {
      if constexpr (std::is_same<T, double>::value)
        hipLaunchKernelGGL((k_aux<T, 0, false>), grid, dim3(kBlock), 0, s, sc, b, band_first, sb, stats);
    } else {
      auto aux = [&](auto deep_tag) {
        constexpr bool D = decltype(deep_tag)::value;
        if (formula == 7)
          hipLaunchKernelGGL((k_aux<T, 7, D>), grid, dim3(kBlock), 0, s, sc, b, band_first, sb, stats);
        else if (formula == 8)
          hipLaunchKernelGGL((k_aux<T, 8, D>), grid, dim3(kBlock), 0, s, sc, b, band_first, sb, stats);
        else
          hipLaunchKernelGGL((k_aux<T, 2, D>), grid, dim3(kBlock), 0, s, sc, b, band_first, sb, stats);
      };
      if (deep) aux(std::true_type{});
      else aux(std::false_type{});
    }
  }
  if (ev_ao0) {
    hipError_t e = hipEventRecord(ev_ao0, s);
    if (e != hipSuccess) return e;
  }
  if (sbuf.slow_ao) {
    if (deep)
      march_variant(formula, 0, false, [&](auto f, auto, auto) {
        constexpr int F = decltype(f)::value;
        if constexpr (F != 0 && !formula_march64(F)) aok(std::true_type{}, f, std::integral_constant<int, kOptions>{}, std::integral_constant<int, 0>{});
      });
    else
      march_variant(formula, sbuf.plain, sbuf.ip8, [&](auto f, auto pl, auto ip) { aok(std::false_type{}, f, pl, ip); });
  }
  if (ev_ao1) {
    hipError_t e = hipEventRecord(ev_ao1, s);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((k_compose<T, T>), grid, dim3(kBlock), 0, s, sc, b, band_first, ao, sb, ended);
  return hipGetLastError();
}
#endif

#if MBR_UNIT(2)
template hipError_t shade_run<double>(const DevScene *, const BandBufs &, int, AODev, ShadeBufs, int,
                                      unsigned long long *, hipStream_t, hipEvent_t, hipEvent_t);
#endif
#if MBR_UNIT(3)
template hipError_t shade_run<float>(const DevScene *, const BandBufs &, int, AODev, ShadeBufs, int,
                                     unsigned long long *, hipStream_t, hipEvent_t, hipEvent_t);
#endif

#if MBR_UNIT(4)
hipError_t launch_shade(int precision, const DevScene *sc, const BandBufs &b, int band_first, AODev ao,
                        ShadeBufs sbuf, int persist_blocks, unsigned long long *stats, hipStream_t s,
                        hipEvent_t ev_ao0, hipEvent_t ev_ao1) {
  // generic formulas in FP32: FP32_FIXUP without aux lights (the host keeps
  // other generic scenes in FP64)
  if (formula_generic(sbuf.formula) && (precision > 1 || (precision == 1 && sbuf.lights))) return hipErrorInvalidValue;
  if (precision == 0) return shade_run<double>(sc, b, band_first, ao, sbuf, persist_blocks, stats, s, ev_ao0, ev_ao1);
  return shade_run<float>(sc, b, band_first, ao, sbuf, persist_blocks, stats, s, ev_ao0, ev_ao1);
}

hipError_t launch_finish(int precision, const DevScene *sc, const BandBufs &b, int band_first, int band_rays,
                         FrameOut out, hipStream_t s, int formula, int fx, int vis, int persist_blocks,
                         unsigned long long *stats, AODev ao) {
  if (band_rays <= 0) return hipSuccess;
  if (fx) {
    if (formula_generic(formula) && precision != 0) return hipErrorInvalidValue;
    const dim3 grid((unsigned)std::max(1, std::min(persist_blocks, (band_rays + kBlock - 1) / kBlock)));
    if (formula_generic(formula)) {
      hipLaunchKernelGGL((k_finish_fx<double, double, 0>), grid, dim3(kBlock), 0, s, sc, b, band_first, band_rays,
                         out, stats, ao);
      return hipGetLastError();
    }
    auto run = [&](auto tag, auto rtag) {
      using T = decltype(tag);
      using RT = decltype(rtag);
      if (formula == 7)
        hipLaunchKernelGGL((k_finish_fx<T, RT, 7>), grid, dim3(kBlock), 0, s, sc, b, band_first, band_rays, out,
                           stats, ao);
      else if (formula == 8)
        hipLaunchKernelGGL((k_finish_fx<T, RT, 8>), grid, dim3(kBlock), 0, s, sc, b, band_first, band_rays, out,
                           stats, ao);
      else
        hipLaunchKernelGGL((k_finish_fx<T, RT, 2>), grid, dim3(kBlock), 0, s, sc, b, band_first, band_rays, out,
                           stats, ao);
    };
    if (precision == 0) run(double{}, double{});
    else run(float{}, float{});
    return hipGetLastError();
  }
  auto plain = [&](auto tag, auto vis_tag) {
    using T = decltype(tag);
    constexpr bool V = decltype(vis_tag)::value;
    hipLaunchKernelGGL((k_finish<T, T, V>), grid_for(band_rays), dim3(kBlock), 0, s, sc, b, band_first, band_rays,
                       out);
  };
  if (precision == 0) {
    if (vis) plain(double{}, std::true_type{});
    else plain(double{}, std::false_type{});
  } else {
    if (vis) plain(float{}, std::true_type{});
    else plain(float{}, std::false_type{});
  }
  return hipGetLastError();
}
#endif  // finish

}  // namespace mbr
