"""The buffer that FastAmbientOcclusion2's estimates are kept in: it has the
size of the frame, not of the largest band, and a render that cannot have it
sums each hit's estimates one after the other instead of failing (same AO: the
sums run in the same order)."""
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

from mandelbulber_amd import _abi, scene

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
W, H, QUALITY = 96, 64, 8


def _scene(fast, formula=7):
    s = scene.menger_view(W, H, shaded=False)
    s.formula = formula
    return scene.apply(s, {"ambient_occlusion_enabled": fast, "fast_ambient_occlusion_mode": 1,
                           "ambient_occlusion_quality": QUALITY})


@pytest.mark.parametrize("formula,prec", [(7, _abi.PREC_FP64), (7, _abi.PREC_FP32_FIXUP), (17, _abi.PREC_FP64)])
def test_fast_ao_memory_follows_the_frame(formula, prec):
    import torch
    from mandelbulber_amd import Renderer
    r = Renderer(0)
    r.set_scene(_scene(0, formula))
    r.render(precision=prec)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    r.set_scene(_scene(1, formula))
    r.render(precision=prec)
    torch.cuda.synchronize()
    grown = before - torch.cuda.mem_get_info()[0]
    r.close()
    # the estimates of a 96x64 frame's hits take 3.1 MB at most; device memory
    # is handed out in pieces of 2 MB and more
    print(f"[fast AO] formula {formula} precision {prec}: {grown / 2**20:.1f} MiB", flush=True)
    assert grown <= 64 * 2**20


# hipMalloc of the sizes in MBR_TEST_FAIL_SIZES finds no memory
SHIM = r"""
#include <cstdlib>
#include <cstring>
#include <cstdio>
#include <dlfcn.h>
extern "C" int hipMalloc(void **p, size_t n) {
  static auto real = (int (*)(void **, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), "hipMalloc");
  char size[32];
  std::snprintf(size, sizeof size, ",%zu,", n);
  const char *list = std::getenv("MBR_TEST_FAIL_SIZES");
  if (list && std::strstr(list, size)) {
    std::printf("refused %zu\n", n);
    std::fflush(stdout);
    return 2;  // hipErrorOutOfMemory
  }
  return real(p, n);
}
"""

CHILD = r"""
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
sys.path.insert(0, sys.argv[2])
sys.path.insert(0, sys.argv[2] + "/tests")
from mandelbulber_amd import Renderer
import test_gpu_fast_ao_memory as T
r = Renderer(0)
r.set_scene(T._scene(1))
f, st = r.render(precision=int(sys.argv[3]))
np.savez(sys.argv[4], rgb=f.rgb, z=f.z, hits=st.hits)
r.close()
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("prec", [_abi.PREC_FP64, _abi.PREC_FP32_FIXUP])
def test_fast_ao_without_its_buffer(tmp_path, prec):
    src, so = tmp_path / "shim.cpp", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(src), "-o", str(so), "-ldl"], check=True)
    values, size = QUALITY * QUALITY - 1, 8 if prec == _abi.PREC_FP64 else 4
    # of the frame's hits, and of the largest band's
    sizes = f",{W * H * values * size},{(1 << 21) * values * size},"
    frames = []
    for fail in ("", sizes):
        out = tmp_path / f"out{len(frames)}.npz"
        env = dict(os.environ, MBR_TEST_FAIL_SIZES=fail)
        r = subprocess.run([sys.executable, "-c", CHILD, str(so), ROOT, str(prec), str(out)], env=env,
                           capture_output=True, text=True, timeout=100)
        print(r.stdout, r.stderr[-2000:], flush=True)
        assert r.returncode == 0, r.stderr[-2000:]
        assert ("refused" in r.stdout) == bool(fail)
        frames.append(np.load(out))
    assert frames[0]["hits"] > 0
    assert np.array_equal(frames[0]["z"], frames[1]["z"])
    assert np.array_equal(frames[0]["rgb"], frames[1]["rgb"])
