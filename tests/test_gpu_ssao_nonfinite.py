"""SSAO on depth planes with samples that have no slope: infinite, NaN, huge,
zero, negative and equal depths among ordinary ones.  The GPU compares samples
by cross products, the reference by quotients (src/image.cpp:335-360); the
16-bit results hold the bar of the ordinary planes."""
import numpy as np
import pytest

from mandelbulber_amd import scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("special", [-np.inf, np.inf, np.nan, 3e38, -3e38, 1e-38, 0.0, -2.5])
@pytest.mark.parametrize("ptype", [0, 1, 2])
def test_ssao_special_depths(ptype, special):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible GPU")
    from mandelbulber_amd import Renderer
    from oracle import oracle
    w, h = 96, 64
    rng = np.random.default_rng(5)
    z = (2.5 + 0.5 * rng.random((h, w))).astype(np.float32)
    z[rng.random((h, w)) < 0.3] = 2.75
    z[rng.random((h, w)) < 0.1] = 1e20
    z[rng.random((h, w)) < 0.05] = special
    s = scene.mandelbulb_plain(w, h)
    s.perspective_type, s.ssao_quality = ptype, 9
    op = rng.integers(0, 30000, (h, w)).astype(np.uint16)
    col = rng.integers(0, 256, (3, h, w)).astype(np.uint8)
    img = rng.integers(0, 30000, (h, w, 3)).astype(np.uint16)
    want = oracle.ssao(s, z, op, col, img)
    r = Renderer(0)
    got = r.post_ssao(s, z, op, col, img.copy())
    r.close()
    # a special centre's own horizon may be undefined (its bytes are then a
    # conversion of NaN); every other pixel holds the bar
    centre = ~((z == special) | np.isnan(z))
    d = np.abs(got.astype(np.int32) - want.astype(np.int32))[centre]
    print(f"[ssao] perspective {ptype} depth {special}: max diff {d.max()}, {np.count_nonzero(d)} of {d.size}", flush=True)
    assert d.max() <= 1 and np.count_nonzero(d) <= 1e-4 * d.size + 1
