"""The depth-of-field splat order (dof_order): sort and shuffle against a plain
restatement of PostRendering_DOF's order (src/image.cpp:57-152,
src/common_math.h:53-84) compiled beside it, for planes with ties, both sides of
the focus, sizes beyond FP32's range and images small enough for every draw to
be a last one.  Ranks are equal."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include <cmath>
#include <cstdio>
#include <cstdint>
#include <vector>
#include "mbr_rand.hpp"
namespace mbr {
void dof_order(const float *z, int w, int h, double neutral, double deep, uint32_t seed, uint32_t *rank);
}
struct E { float z; int i; };
static void qs(std::vector<E> &d, int l, int p) {
  int i = l, j = p;
  const float x = d[(l + p) / 2].z;
  do {
    while (d[i].z < x) i++;
    while (x < d[j].z) j--;
    if (i <= j) { E t = d[i]; d[i] = d[j]; d[j] = t; i++; j--; }
  } while (i <= j);
  if (l < j) qs(d, l, j);
  if (i < p) qs(d, i, p);
}
static void order(const float *z, int n, double neutral, double deep, uint32_t seed, uint32_t *rank) {
  std::vector<E> d(n);
  for (int k = 0; k < n; k++) d[k] = {z[k], k};
  if (n > 2) qs(d, 1, n - 1);
  mbr::GlibcRand rnd(seed);
  for (int i = n - 1; i >= 0; i--) {
    const E t = d[i];
    const double z1 = t.z, s1 = (z1 - neutral) / z1 * deep;
    int step = i, ii;
    bool done;
    do {
      ii = i - rnd.next() % (step + 1);
      if (ii <= 0) ii = 0;
      const double z2 = d[ii].z, s2 = (z2 - neutral) / z2 * deep;
      done = false;
      if (s1 * s2 > 0) done = (s1 > 0 ? s2 / s1 : s1 / s2) > 0.7;
      step = (int)(step * 0.7 - 1);
      if (step <= 0) done = true;
    } while (!done);
    d[i] = d[ii];
    d[ii] = t;
  }
  for (int k = 0; k < n; k++) rank[d[n - 1 - k].i] = k;
}
int main() {
  int bad = 0;
  for (int c = 0; c < 12; c++) {
    const int w = c < 4 ? 1 + c * 3 : 37 * c, h = c < 4 ? 1 + c : 29 + 13 * c, n = w * h;
    std::vector<float> z(n);
    mbr::GlibcRand r(c + 1);
    for (int k = 0; k < n; k++) {
      const double u = r.next() / 2147483648.0;
      z[k] = u < 0.3 ? 1e20f : (float)(c % 3 == 0 ? std::floor(40 * u) / 10 : 2.0 + 2.0 * u);
      if (c == 7 && u > 0.99) z[k] = 2.7f;
      if (c == 8 && u > 0.9) z[k] = (float)(1e-25 * u);
    }
    std::vector<uint32_t> a(n), b(n);
    const double deep = c == 9 ? 1e19 : c == 10 ? 1e-22 : 6.0;
    mbr::dof_order(z.data(), w, h, 2.7, deep, 100 + c, a.data());
    order(z.data(), n, 2.7, deep, 100 + c, b.data());
    if (a != b) { std::printf("case %d (%d pixels) differs\n", c, n); bad++; }
  }
  return bad;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_dof_order_equals_restatement(tmp_path):
    src = tmp_path / "check.cpp"
    src.write_text(CHECK)
    exe = tmp_path / "check"
    csrc = os.path.join(ROOT, "mandelbulber_amd", "csrc")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include", f"-I{csrc}",
                    f"-I{ROOT}/include", str(src), os.path.join(csrc, "mbr_post_order.cpp"), "-o", str(exe),
                    "-lpthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
