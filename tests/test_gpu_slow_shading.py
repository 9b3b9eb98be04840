"""slowShading's 11^3 normal stencil (src/shaders.cpp:720-757), a wave per hit
and a lane per estimate, against the oracle: equal in FP64 for the folding
formulas, whose arithmetic is the oracle's, with and without options, in frames
of few hits and of more hits than waves; and not slower than the same frame
shaded by as many estimates one after the other on a lane would be (it took 14
ms so, against 1.4)."""
import time

import pytest

from mandelbulber_amd import _abi, scene
from metrics import assert_parity, assert_planes_exact, compare

pytestmark = pytest.mark.gpu

VIEWS = {"box": scene.mandelbox_view, "menger": scene.menger_view}


@pytest.fixture(scope="module")
def renderer():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible GPU")
    from mandelbulber_amd import Renderer
    r = Renderer(0)
    yield r
    r.close()


@pytest.mark.parametrize("kind,w,h,keys", [("menger", 5, 4, {}), ("box", 96, 72, {"N": 12}),
                                           ("box", 33, 21, {"N": 12, "interior_mode": 1}),
                                           ("menger", 33, 21, {"limits_enabled": 1, "x_min": -0.45, "z_min": -0.8})])
def test_slow_shading_matches_oracle(renderer, kind, w, h, keys):
    from oracle import oracle
    s = VIEWS[kind](w, h, shaded=False)
    scene.apply(s, dict(keys, slow_shading=1))
    print(f"[slow shading] {kind} {w}x{h} {keys}", flush=True)
    ref, ost = oracle.render(s)
    renderer.set_scene(s)
    f, st = renderer.render(precision=_abi.PREC_FP64)
    m = compare(f, ref)
    print(f"  {st.hits} hits {m}", flush=True)
    assert st.hits > 0 and m["flips"] == 0 and m["psnr_db"] >= 120, m
    assert st.iterations == ost.iterations  # (calls that end without iterating are counted by the GPU only)
    assert_planes_exact(m)
    fix, _ = renderer.render(precision=_abi.PREC_FP32_FIXUP)
    assert_parity(compare(fix, ref), label="fixup")


def test_slow_shading_is_not_a_chain(renderer):
    s = scene.mandelbulb_plain(120, 90)
    scene.apply(s, {"slow_shading": 1, "N": 30})
    renderer.set_scene(s)
    best = 1e9
    for _ in range(5):
        t = time.perf_counter()
        renderer.render(precision=_abi.PREC_FP64)
        best = min(best, time.perf_counter() - t)
    print(f"[slow shading] 120x90 FP64 bulb: {best * 1e3:.2f} ms", flush=True)
    assert best < 9e-3
