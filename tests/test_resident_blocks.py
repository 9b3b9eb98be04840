"""The size of the persistent launches follows the device they go to: two
devices of different CU counts in one process each get their own (the HIP
runtime's answers are made up here)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

CHECK = r"""
#include <cstdio>
#include "mbr_lanes.hpp"
static int device = 0, asked = 0;
extern "C" hipError_t hipGetDevice(int *d) { *d = device; return hipSuccess; }
extern "C" hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int d) {
  *v = d == 0 ? 256 : d == 1 ? 64 : d;
  return hipSuccess;
}
extern "C" hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  asked++;
  *n = 4;
  return device == 3 ? hipErrorInvalidValue : hipSuccess;
}
int main() {
  static std::atomic<int> known[mbr::kKnownDevices];
  const int devices[] = {0, 1, 0, 1, 2, 3, 40, 0}, want[] = {1024, 256, 1024, 256, 8, 1 << 20, 160, 1024};
  int bad = 0;
  for (int i = 0; i < 8; i++) {
    device = devices[i];
    const int n = mbr::resident_blocks((const void *)main, known);
    if (n != want[i]) { std::printf("device %d: %d, want %d\n", device, n, want[i]); bad++; }
  }
  if (asked != 5) { std::printf("asked %d times\n", asked); bad++; }
  return bad;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_resident_blocks_per_device(tmp_path):
    src, exe = tmp_path / "check.hip", tmp_path / "check"
    src.write_text(CHECK)
    csrc = os.path.join(ROOT, "mandelbulber_amd", "csrc")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I" + csrc,
                    "-I" + os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True, capture_output=True,
                   timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
