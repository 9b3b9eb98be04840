"""The FP64 march kernel (march and binary search in one state machine) where
its dispatch and its lane hand-out can go wrong, against the oracle: frames of
fewer rays than a wave, ragged ones, the rotated and the unrotated Mandelbox,
and a coarse quality (a wide search band).  (Refined hits, which the oracle
does not have, are covered by the adjoint's finite differences.)
FP64 frames equal the oracle's depths and integer planes; FP32_FIXUP marches in FP64, so its depths equal those of the
FP64 frame where the iteration is the same (Mandelbox, Menger)."""
import numpy as np
import pytest

from mandelbulber_amd import _abi, scene
from metrics import assert_planes_exact, compare

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def renderer():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible GPU")
    from mandelbulber_amd import Renderer
    r = Renderer(0)
    yield r
    r.close()


BOX_ROTATED = {"mandelbox_rotation_enabled": 1, "mandelbox_rotation_main_alfa": 10, "mandelbox_rotation_X1_alfa": 7,
               "mandelbox_rotation_Y2_beta": 12}

CASES = [
    ("bulb", 1, 1, {}), ("box", 3, 1, {}), ("menger", 65, 2, {}), ("bulb", 63, 5, {}), ("box", 129, 33, {}),
    ("menger", 97, 41, {"quality": 60}), ("box", 97, 41, {"quality": 60}), ("box", 97, 41, BOX_ROTATED),
    ("box", 97, 41, {"minN": 3}),
]


@pytest.mark.parametrize("kind,w,h,keys", CASES)
def test_march_matches_oracle(renderer, kind, w, h, keys):
    from oracle import oracle
    s = {"bulb": scene.mandelbulb_plain, "box": lambda a, b: scene.mandelbox_view(a, b, shaded=False),
         "menger": lambda a, b: scene.menger_view(a, b, shaded=False)}[kind](w, h)
    scene.apply(s, keys)
    print(f"[march] {kind} {w}x{h} {keys}", flush=True)
    ref, _ = oracle.render(s)
    renderer.set_scene(s)
    f64, st = renderer.render(precision=_abi.PREC_FP64)
    m = compare(f64, ref)
    print(f"  {m}", flush=True)
    assert st.hits == int(np.count_nonzero(f64.z < 1e19))
    if keys is BOX_ROTATED:
        # rotations round fused here and apart in the oracle
        assert m["flip_frac"] <= 1e-3 and m["depth_rel_max"] <= 1e-4, m
    else:
        assert m["flips"] == 0 and m["depth_rel_max"] <= 1e-12, m
        assert_planes_exact(m)
    fix, _ = renderer.render(precision=_abi.PREC_FP32_FIXUP)
    if kind != "bulb":
        np.testing.assert_array_equal(fix.z, f64.z)
    m = compare(fix, ref)
    assert m["flip_frac"] <= 1e-3 and m["depth_rel_max"] <= 1e-4, m
