// mbr_adjoint.hip — gradient of a pixel loss with respect to the scene
// parameters (formula power, camera position and angles, light angles) for
// FP64 Mandelbulb renders with refined hits (mbr_scene.hit_refine = 1).
//
// The caller supplies the adjoint of the image, dL/dC for every pixel and
// channel.  The kernel returns sum_pixels sum_channels dL/dC . dC/dtheta for
// the nine parameters theta = (power, vp x/y/z, alfa, beta, gamma, light
// alfa, light beta): a vector-Jacobian product, formed per pixel from the
// nine tangents of the pixel's colour, then reduced over the image.
//
// What the colour of a pixel depends on, in the order of the forward:
//   camera: R = Rz(alfa) Rx(beta) Ry(gamma) (src/algebra.cpp:94-143), ray
//     start o = vp - R (0, zoom/persp, 0), view vector d = R (x2 fov, 1, z2 fov)
//     (src/Render3D.cpp:316-333, :389-438);
//   hit: the refined hit t solves F(t) = D(o + t d; power) - c0 thr(t) = 0
//     with thr(t) = t res persp / quality and c0 = 1 - 0.005 quality, so by
//     the implicit function theorem dt = -(dD/dtheta at fixed t) / (dD/dt -
//     c0 dthr/dt), and the hit point p = o + t d moves by do + t dd + d dt;
//   normal: forward differences of D at p (N x 5 iterations, minN 0) with the
//     step delta = thr quality smoothness (src/shaders.cpp:675-757), each
//     distance estimate carrying its gradient in (p, power);
//   light L = R (cos(aL - pi/2) cos(-bL), sin(aL - pi/2) cos(-bL), sin(-bL))
//     (src/Render3D.cpp:253-256);
//   shading: main light x direct light x ((1 - shading) + shading max(0,
//     n.L)) x colour + main light x specular min(15, max(0, n.h)^30) with h =
//     normalize(L - d) (ObjectShader, src/shaders.cpp:21-112); shadows, AO,
//     glow and fog are rejected by mbr_adjoint;
//   misses: the background gradient on d.(0,0,-1) (src/shaders.cpp:159-181).
// The surface colour is an integer palette index (floor of the orbit value,
// src/shaders.cpp:855-870) and the background is stored as 16-bit integers:
// both are steps in theta whose derivative is zero almost everywhere; the
// kernel uses zero for the colour and the slope of the gradient before the
// 16-bit rounding for the background.  Pixels whose depth or normal is
// ill-conditioned (grazing hits, degenerate normals) are left out.
#include "mbr_kernels.hpp"
#include "mbr_lanes.hpp"
#include "mbr_shade.hpp"

namespace mbr {

constexpr int kParams = 9;
constexpr double kTangentMax = 1e5;
// residual of a refined hit, relative to its threshold, below which it
// counts as a root of F (the refinement stops at 1e-13)
constexpr double kRootTol = 1e-7;

// Value and gradient in (p.x, p.y, p.z, power).
struct G4 {
  double v, g[4];
};

// CalculateDistance of the trig_optim Mandelbulb (src/fractal.cpp:211-225,
// :1151-1157, :1245-1306 for the analytic branch without interior mode,
// iteration threshold, primitives or limits) with its gradient in (point,
// power), as a resumable state; the branches follow the values, as in the
// forward.  An iteration forms its transcendentals once and carries the four
// tangent columns of the orbit and of its derivative through their slopes.
struct GradDE {
  V3<double> z, c, dz[4];
  double r, aux, dr[4], daux[4];
  int L;

  __device__ __forceinline__ void begin(const FractalK<double> &f, V3<double> p) {
    z = p;
    c = f.julia_mode ? v3<double>(f.julia[0], f.julia[1], f.julia[2]) : p * f.constant_factor;
    r = length(z);
    aux = 1.0;
    L = 0;
    for (int i = 0; i < 4; i++) {
      dz[i] = v3<double>(i == 0, i == 1, i == 2);
      dr[i] = r > 0 ? dot(z, dz[i]) / r : 0.0;
      daux[i] = 0.0;
    }
  }
  // one iteration; true when the orbit escaped (L < N) or N is reached
  __device__ __forceinline__ bool step(const FractalK<double> &f, double power, int N) {
    const double u = z.z / r, th0 = asin(u), ph0 = atan2(z.y, z.x);
    const double rp = radius_power(f, r), lr = log(r);
    double sth, cth, sph, cph;
    sincos(th0 * power, &sth, &cth);
    sincos(ph0 * power, &sph, &cph);
    const double dasin = 1.0 / sqrt(1.0 - u * u), ir = 1.0 / r;
    const double den = z.x * z.x + z.y * z.y;
    const double ix = den > 0 ? z.x / den : 0.0, iy = den > 0 ? z.y / den : 0.0;
    const double drp = (power - 1.0) * rp * ir;  // d rp / dr
    const double R = rp * r;
    const double k = f.julia_mode ? 0.0 : f.constant_factor;
    const V3<double> e = v3<double>(cth * cph, cth * sph, sth);
    const V3<double> zn = e * R + c;
    const double rn = length(zn), irn = rn > 0 ? 1.0 / rn : 0.0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const double dp = i == 3 ? 1.0 : 0.0;
      const double du = (dz[i].z - u * dr[i]) * ir;
      const double dth = du * dasin * power + th0 * dp;
      const double dph = (ix * dz[i].y - iy * dz[i].x) * power + ph0 * dp;
      const double dr1 = drp * dr[i] + rp * lr * dp;
      daux[i] = (dr1 * aux + rp * daux[i]) * power + rp * aux * dp;
      const double dR = dr1 * r + rp * dr[i];
      const V3<double> dn =
          v3<double>(R * (-sth * cph * dth - e.y * dph) + e.x * dR + (i == 0 ? k : 0.0),
                     R * (-sth * sph * dth + e.x * dph) + e.y * dR + (i == 1 ? k : 0.0),
                     R * (cth * dth) + sth * dR + (i == 2 ? k : 0.0));
      dz[i] = dn;
      dr[i] = dot(zn, dn) * irn;
    }
    aux = rp * aux * power + 1.0;
    z = zn;
    r = rn;
    if (!(r <= f.bailout)) return true;
    L++;
    return L >= N;
  }
  __device__ __forceinline__ G4 end(double detail, int N, int minN) const {
    G4 d = {0.0, {0, 0, 0, 0}};
    if (L < N) {
      const double lr = log(r);
      d.v = r * lr * 0.5 / aux;
      const double ia = 1.0 / aux;
      for (int i = 0; i < 4; i++) d.g[i] = ((lr + 1.0) * dr[i] * 0.5 - d.v * daux[i]) * ia;
    }
    if (d.v < 0) d = G4{0.0, {0, 0, 0, 0}};
    if (L < minN && d.v < detail) d = G4{detail, {0, 0, 0, 0}};
    return d;
  }
};

// Rotation Rz(a) Rx(b) Ry(g) and its derivatives in a, b, g (row-major).
__device__ void rot3(double a, double b, double g, double R[9], double dR[3][9]) {
  const double ca = cos(a), sa = sin(a), cb = cos(b), sb = sin(b), cg = cos(g), sg = sin(g);
  const double Z[9] = {ca, -sa, 0, sa, ca, 0, 0, 0, 1}, dZ[9] = {-sa, -ca, 0, ca, -sa, 0, 0, 0, 0};
  const double X[9] = {1, 0, 0, 0, cb, -sb, 0, sb, cb}, dX[9] = {0, 0, 0, 0, -sb, -cb, 0, cb, -sb};
  const double Y[9] = {cg, 0, sg, 0, 1, 0, -sg, 0, cg}, dY[9] = {-sg, 0, cg, 0, 0, 0, -cg, 0, -sg};
  auto mul3 = [](const double *A, const double *B, const double *C, double *out) {
    double t[9];
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) t[i * 3 + j] = A[i * 3] * B[j] + A[i * 3 + 1] * B[3 + j] + A[i * 3 + 2] * B[6 + j];
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) out[i * 3 + j] = t[i * 3] * C[j] + t[i * 3 + 1] * C[3 + j] + t[i * 3 + 2] * C[6 + j];
  };
  mul3(Z, X, Y, R);
  mul3(dZ, X, Y, dR[0]);
  mul3(Z, dX, Y, dR[1]);
  mul3(Z, X, dY, dR[2]);
}

__device__ __forceinline__ V3<double> mv(const double *M, const V3<double> &v) {
  return v3<double>(M[0] * v.x + M[1] * v.y + M[2] * v.z, M[3] * v.x + M[4] * v.y + M[5] * v.z,
                    M[6] * v.x + M[7] * v.y + M[8] * v.z);
}

// d/dtheta of normalize(v), given v and its tangent dv
__device__ __forceinline__ V3<double> dnormalize(const V3<double> &v, const V3<double> &dv) {
  const double l = length(v);
  const V3<double> u = v * (1.0 / l);
  return (dv - u * dot(u, dv)) * (1.0 / l);
}

// The estimates with gradients of the band's hits, in planes over the band's
// rays: value and four slopes of estimate j at [(5 j + i) cap + r], j = 0 at the
// hit (the implicit equation), 1..4 the normal's stencil.
__device__ __forceinline__ G4 load_g4(const double *g4, long long cap, int j, int r) {
  const double *q = g4 + 5 * j * cap + r;
  return G4{q[0], {q[cap], q[2 * cap], q[3 * cap], q[4 * cap]}};
}

// Whether the hit's depth has a derivative here.  It is well conditioned where
// the ray meets the level set D = c0 thr going down it: Ft = dF/dt < 0 with a
// margin.  Near a grazing tangency Ft -> 0 and dt/dtheta diverges: the refined
// hit then sits next to a fold of t(theta), where the forward jumps for a small
// change of theta.  The implicit-function derivative holds at a root of F;
// where the distance estimate jumps across the binary search's band (its
// spherical coordinates are singular on the z axis and its preimages) the
// refinement stops short of a root, and the depth then follows the Newton
// iterates instead.  Both kinds of hits are left out (and flagged).
__device__ __forceinline__ bool has_root(const G4 &D, const V3<double> &d, double thr, double c0, double kthr,
                                         double &Ft) {
  const V3<double> gD = v3<double>(D.g[0], D.g[1], D.g[2]);
  Ft = dot(gD, d) - c0 * kthr;
  return Ft < -0.05 * length(gD) * length(d) && fabs(D.v - c0 * thr) <= kRootTol * thr;
}

// The hits' estimates, one per lane and item (mbr_lanes.hpp); Stencil: the
// normal's, of the hits that have a root.  Five estimates after one another per
// lane, the stencil's with 5 N iterations, left a 512x512 image waiting for the
// few lanes whose orbits never escape (7.5 ms of 256-register kernel).
template <bool Stencil>
__global__ void __launch_bounds__(kBlock, 2)
    k_adjoint_de(const DevScene *__restrict__ scp, BandBufs b, int band_first, AdjParams P,
                 const float *__restrict__ gR, const float *__restrict__ gG, const float *__restrict__ gB, bool all,
                 double *__restrict__ g4) {
  const DevScene &sc = *scp;
  const FractalK<double> f = sc.fd;
  const ShadeK<double> &k = sc.sd;
  const double kthr = k.resolution * k.persp / k.quality, c0 = 1.0 - 0.005 * k.quality;
  const long long n_items = (long long)b.counters[CNT_HITS] * (Stencil ? 4 : 1);
  const int N = Stencil ? sc.N * 5 : sc.N, minN = Stencil ? 0 : sc.minN;
  const int lanes = item_lanes(n_items);
  WaveQueue<> queue(&b.counters[Stencil ? CNT_NORMALQ : CNT_SHADOWQ], n_items, lanes);
  const int lane = __lane_id();
  int state = lane < lanes ? MS_NEED : MS_EXHAUSTED;
  int r = 0, j = 0;
  double thr = 0;
  GradDE de;
  lane_loop<2>(
      state,
      [&](int rank, int n_need) {
        const long long mine = queue.take(b, rank, n_need);
        if (state != MS_NEED) return;
        if (mine < 0) {
          state = MS_EXHAUSTED;
          return;
        }
        r = b.hit_list[Stencil ? mine >> 2 : mine];
        j = Stencil ? 1 + (int)(mine & 3) : 0;
        const int p = band_first + r;
        if (!all && gR[p] == 0.0f && gG[p] == 0.0f && gB[p] == 0.0f) return;
        thr = b.thr[r];
        V3<double> q = v3<double>(b.px[r], b.py[r], b.pz[r]);
        if constexpr (Stencil) {
          V3<double> d;
          view_vector(sc, p % sc.width, p / sc.width, d);
          double Ft;
          if (!has_root(load_g4(g4, b.cap, 0, r), d, thr, c0, kthr, Ft)) return;
          const double delta = thr * k.quality * k.smoothness;
          q = q + v3<double>(j == 2 ? delta : 0.0, j == 3 ? delta : 0.0, j == 4 ? delta : 0.0);
        }
        de.begin(f, q);
        state = MS_ITER;
      },
      [&]() { return de.step(f, P.power, N); },
      [&]() {
        const G4 D = de.end(thr, N, minN);
        double *o = g4 + 5 * j * (long long)b.cap + r;
        o[0] = D.v;
        for (int i = 0; i < 4; i++) o[(i + 1) * (long long)b.cap] = D.g[i];
        state = MS_NEED;
      });
}

// Per pixel: the nine tangents of its colour, contracted with the image adjoint.
__global__ void __launch_bounds__(kBlock) k_adjoint(const DevScene *__restrict__ scp, BandBufs b, int band_first,
                                                    int band_rays, AdjParams P, const float *__restrict__ gR,
                                                    const float *__restrict__ gG, const float *__restrict__ gB,
                                                    double *grad, uint8_t *skipped, float *__restrict__ jac,
                                                    const double *__restrict__ g4) {
  const DevScene &sc = *scp;
  const ShadeK<double> &k = sc.sd;
  double acc[kParams];
  for (int i = 0; i < kParams; i++) acc[i] = 0;
  double R[9], dR[3][9];
  rot3(P.alpha, P.beta, P.gamma, R, dR);
  // light: L = R lv(aL, bL)
  const V3<double> lv = v3<double>(cos(P.light_alpha - 0.5 * M_PI) * cos(-P.light_beta),
                                   sin(P.light_alpha - 0.5 * M_PI) * cos(-P.light_beta), sin(-P.light_beta));
  const V3<double> dlv_a = v3<double>(-sin(P.light_alpha - 0.5 * M_PI) * cos(-P.light_beta),
                                      cos(P.light_alpha - 0.5 * M_PI) * cos(-P.light_beta), 0.0);
  const V3<double> dlv_b = v3<double>(cos(P.light_alpha - 0.5 * M_PI) * sin(-P.light_beta),
                                      sin(P.light_alpha - 0.5 * M_PI) * sin(-P.light_beta), -cos(-P.light_beta));
  const V3<double> L = mv(R, lv);
  V3<double> dL[kParams];
  for (int i = 0; i < kParams; i++) dL[i] = v3<double>(0, 0, 0);
  for (int a = 0; a < 3; a++) dL[4 + a] = mv(dR[a], lv);
  dL[7] = mv(R, dlv_a);
  dL[8] = mv(R, dlv_b);
  const V3<double> yz = v3<double>(0.0, P.zoom_persp, 0.0);  // start = vp - R (0, zoom/persp, 0)
  const double kthr = k.resolution * k.persp / k.quality;
  const double c0 = 1.0 - 0.005 * k.quality;
  const double mlR = k.main_light[0], mlG = k.main_light[1], mlB = k.main_light[2];

  for (long long rr = (long long)blockIdx.x * kBlock + threadIdx.x; rr < band_rays;
       rr += (long long)gridDim.x * kBlock) {
    const int r = (int)rr;
    const int p = band_first + r;
    const int x = p % sc.width, y = p / sc.width;
    const size_t npix = (size_t)sc.width * sc.height;
    const double aR = jac ? 0.0 : gR[p], aG = jac ? 0.0 : gG[p], aB = jac ? 0.0 : gB[p];
    if (!jac && aR == 0.0 && aG == 0.0 && aB == 0.0) continue;
    if (jac)
      for (int i = 0; i < 3 * kParams; i++) jac[(size_t)i * npix + p] = 0.0f;
    const double x2 = ((double)x / sc.width - 0.5) * sc.aspect;
    const double z2 = (double)y / sc.height - 0.5;
    const V3<double> v0 = v3<double>(x2 * sc.fov, 1.0, z2 * sc.fov);
    V3<double> d;  // the forward's view vector (its values); tangents from rot3
    view_vector(sc, x, y, d);
    V3<double> dd[kParams], dO[kParams];
    for (int i = 0; i < kParams; i++) {
      dd[i] = v3<double>(0, 0, 0);
      dO[i] = v3<double>(0, 0, 0);
    }
    for (int a = 0; a < 3; a++) {
      dd[4 + a] = mv(dR[a], v0);
      dO[4 + a] = mv(dR[a], yz) * -1.0;
    }
    if (skipped) skipped[p] = 0;
    dO[1] = v3<double>(1, 0, 0);
    dO[2] = v3<double>(0, 1, 0);
    dO[3] = v3<double>(0, 0, 1);
    double dC[3][kParams];
    if (!b.found[r]) {
      // background gradient on the view vector (src/shaders.cpp:159-181)
      const double grad = -d.z + 1.0;
      for (int i = 0; i < kParams; i++) {
        const double dg = -dd[i].z;
        for (int ch = 0; ch < 3; ch++) {
          const double c1 = sc.bg1[ch], c2 = sc.bg2[ch], c3 = sc.bg3[ch];
          const double slope = grad < 1 ? (c2 - c3) : (c1 - c2);
          dC[ch][i] = slope * dg / 65536.0;
        }
      }
    } else {
      const double t = b.depth[r];
      const V3<double> ph = v3<double>(b.px[r], b.py[r], b.pz[r]);  // the forward's hit point
      const double thr = b.thr[r];
      // the implicit hit
      const G4 D = load_g4(g4, b.cap, 0, r);
      const V3<double> gD = v3<double>(D.g[0], D.g[1], D.g[2]);
      double Ft;
      if (!has_root(D, d, thr, c0, kthr, Ft)) {
        if (skipped) skipped[p] = 1;
        continue;
      }
      if (skipped) skipped[p] = 0;
      double dt[kParams];
      V3<double> dp[kParams];
      for (int i = 0; i < kParams; i++) {
        const double Fi = dot(gD, dO[i] + dd[i] * t) + (i == 0 ? D.g[3] : 0.0);
        dt[i] = fabs(Ft) > 0 ? -Fi / Ft : 0.0;
        dp[i] = dO[i] + dd[i] * t + d * dt[i];
      }
      // normal: forward differences of D at N x 5, minN 0
      const G4 s1 = load_g4(g4, b.cap, 1, r), s2 = load_g4(g4, b.cap, 2, r), s3 = load_g4(g4, b.cap, 3, r),
               s4 = load_g4(g4, b.cap, 4, r);
      const V3<double> nr = v3<double>(s2.v - s1.v, s3.v - s1.v, s4.v - s1.v);
      const bool zero_n = nr.x == 0 && nr.y == 0 && nr.z == 0;
      const V3<double> n = zero_n ? v3<double>(1, 0, 0) : normalize(nr);
      // light and specular (ObjectShader without shadow and ambient terms)
      const double nl = dot(n, L);
      const double shade = k.direct_light * ((1.0 - k.shading) + k.shading * (nl > 0 ? nl : 0.0));
      const V3<double> hr = L - d;
      const V3<double> h = normalize(hr);
      const double nh = dot(n, h);
      const double s2v = nh > 0 ? pow(nh, 30.0) : 0.0;
      const bool spec_live = nh > 0 && s2v < 15.0;
      // colour: the palette index is an integer (derivative zero); the
      // forward's colour, recomputed at the same point
      double col[3] = {1.0, 1.0, 1.0};
      if (sc.coloring) {
        ShaderIn<double> in;
        in.point = ph;
        in.point64 = ph;
        in.detail = thr;
        in.object = b.object[r];
        LaneCount cnt = {0, 0};
        const RGBT<double> colour = surface_colour<double, false, false, 2>(sc, in, cnt);
        col[0] = colour.R;
        col[1] = colour.G;
        col[2] = colour.B;
      }
      for (int i = 0; i < kParams; i++) {
        const double ddelta = k.quality * k.smoothness * kthr * dt[i];
        const V3<double> q = dp[i];
        const double pw = i == 0 ? 1.0 : 0.0;
        const double ds1 = s1.g[0] * q.x + s1.g[1] * q.y + s1.g[2] * q.z + s1.g[3] * pw;
        const double ds2 = s2.g[0] * (q.x + ddelta) + s2.g[1] * q.y + s2.g[2] * q.z + s2.g[3] * pw;
        const double ds3 = s3.g[0] * q.x + s3.g[1] * (q.y + ddelta) + s3.g[2] * q.z + s3.g[3] * pw;
        const double ds4 = s4.g[0] * q.x + s4.g[1] * q.y + s4.g[2] * (q.z + ddelta) + s4.g[3] * pw;
        const V3<double> dnr = v3<double>(ds2 - ds1, ds3 - ds1, ds4 - ds1);
        const V3<double> dn = zero_n ? v3<double>(0, 0, 0) : dnormalize(nr, dnr);
        const double dnl = dot(dn, L) + dot(n, dL[i]);
        const double dshade = nl > 0 ? k.direct_light * k.shading * dnl : 0.0;
        const V3<double> dh = dnormalize(hr, dL[i] - dd[i]);
        const double dnh = dot(dn, h) + dot(n, dh);
        const double dspec = spec_live ? 30.0 * pow(nh, 29.0) * dnh * k.specular : 0.0;
        dC[0][i] = mlR * dshade * col[0] + mlR * dspec;
        dC[1][i] = mlG * dshade * col[1] + mlG * dspec;
        dC[2][i] = mlB * dshade * col[2] + mlB * dspec;
      }
    }
    // A tangent beyond kTangentMax colour units per unit parameter comes from
    // a degenerate normal (the four estimates nearly equal) or a fold of the
    // hit: the pixel is ill-conditioned and left out (and flagged).
    bool finite = true;
    for (int i = 0; i < kParams; i++)
      for (int ch = 0; ch < 3; ch++) finite = finite && fabs(dC[ch][i]) <= kTangentMax;
    if (!finite) {
      if (skipped) skipped[p] = 1;
      continue;
    }
    if (jac) {
      for (int i = 0; i < kParams; i++)
        for (int ch = 0; ch < 3; ch++) jac[(size_t)(i * 3 + ch) * npix + p] = (float)dC[ch][i];
      continue;
    }
    for (int i = 0; i < kParams; i++) acc[i] += aR * dC[0][i] + aG * dC[1][i] + aB * dC[2][i];
  }
  // block reduction, one atomic per parameter and workgroup
  __shared__ double red[kParams][kBlock / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int i = 0; i < kParams; i++) {
    double v = acc[i];
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
    if (lane == 0) red[i][wave] = v;
  }
  __syncthreads();
  if (grad && threadIdx.x < kParams) {
    double v = 0;
    for (int w = 0; w < kBlock / 64; w++) v += red[threadIdx.x][w];
    atomicAdd(&grad[threadIdx.x], v);
  }
}

hipError_t launch_adjoint(const DevScene *sc, const BandBufs &b, int band_first, int band_rays, AdjParams p,
                          const float *gR, const float *gG, const float *gB, double *grad, uint8_t *skipped,
                          float *jac, int blocks, hipStream_t s) {
  if (band_rays <= 0) return hipSuccess;
  if (b.rec_bytes != 8 || b.slab < 25) return hipErrorInvalidValue;
  // the march's step records are not read any more: their planes hold the estimates
  double *g4 = (double *)b.rec_step;
  launch_resident<k_adjoint_de<false>>(blocks, s, sc, b, band_first, p, gR, gG, gB, jac != nullptr, g4);
  launch_resident<k_adjoint_de<true>>(blocks, s, sc, b, band_first, p, gR, gG, gB, jac != nullptr, g4);
  hipLaunchKernelGGL(k_adjoint, dim3(std::max(1, std::min(blocks, (band_rays + kBlock - 1) / kBlock))), dim3(kBlock), 0,
                     s, sc, b, band_first, band_rays, p, gR, gG, gB, grad, skipped, jac, g4);
  return hipGetLastError();
}

}  // namespace mbr
