"""The surface and AO kernels (k_hits, k_fast_ao, k_ao's split hits) where
their hand-out can go wrong, against the oracle: frames with fewer hits than a
wave, ragged ones, AO quality 1 to 3 (several hits per wave) and hits split over
waves, soft shadows, the chained slowShading stencil, FastAmbientOcclusion2.
FP64 frames hold the bars of the parity tests for the same arithmetic (equal
integer planes, 120 dB); FP32_FIXUP frames the parity bars."""
import pytest

from mandelbulber_amd import _abi, scene
from metrics import assert_parity, assert_planes_exact, compare

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


SOFT = {"shadows_enabled": 1, "shadows_cone_angle": 4, "penetrating_lights": 0}
FAST = {"ambient_occlusion_enabled": 1, "fast_ambient_occlusion_mode": 1, "ambient_occlusion_quality": 3}
VIEWS = {"bulb": scene.mandelbulb_plain, "box": lambda w, h: scene.mandelbox_view(w, h, shaded=False),
         "menger": lambda w, h: scene.menger_view(w, h, shaded=False)}

CASES = [("bulb", 5, 3, dict(SOFT, **FAST)), ("box", 7, 5, dict(SOFT, **FAST)), ("menger", 61, 37, dict(SOFT, **FAST)),
         ("box", 19, 13, {"slow_shading": 1}), ("menger", 3, 2, {"slow_shading": 1})]
for _q in (1, 2, 3, 6):
    CASES.append(("box", 21, 17, {"shadows_enabled": 1, "shadows_cone_angle": 0, "ambient_occlusion_enabled": 1,
                                  "ambient_occlusion_quality": _q}))


@pytest.mark.parametrize("kind,w,h,keys", CASES)
def test_shaded_hits_match_oracle(renderer, kind, w, h, keys):
    from oracle import oracle
    s = VIEWS[kind](w, h)
    a, b = scene.light_from_seed(5)
    scene.apply(s, dict(keys, main_light_alfa=a, main_light_beta=b))
    print(f"[hits] {kind} {w}x{h} {keys}", flush=True)
    ref, _ = oracle.render(s)
    renderer.set_scene(s)
    f64, st = renderer.render(precision=_abi.PREC_FP64)
    m = compare(f64, ref)
    print(f"  {st.hits} hits {m}", flush=True)
    assert st.hits > 0 and m["flips"] == 0 and m["depth_rel_max"] <= 1e-12 and m["psnr_db"] >= 120, m
    assert_planes_exact(m)
    fix, _ = renderer.render(precision=_abi.PREC_FP32_FIXUP)
    assert_parity(compare(fix, ref), label="fixup")


@pytest.mark.parametrize("keys", [{"slow_shading": 1, "N": 20}, dict(SOFT, **FAST), {"iter_fog_enabled": 1}])
@pytest.mark.parametrize("formula", [1, 10])
def test_trig_de_and_ifs_hits_match_oracle(renderer, formula, keys):
    """trig_DE and the kaleidoscopic IFS run kernels of their own in plain
    scenes: the chained stencil (FP32 estimates, where the four-point one takes
    FP64 ones), soft shadows with fast AO, and iteration fog (FP64 only)."""
    from oracle import oracle
    if formula == 1:
        s = scene.mandelbulb_plain(31, 23)
        s.power = 8.0
    else:
        s = scene.menger_view(31, 23, shaded=False)
        s.ifs_scale, s.ifs_menger_sponge_mode = 3.0, 1
        for i, d in enumerate([(1, -1, 0), (1, 0, -1), (0, 1, -1)]):
            s.ifs_abs[i], s.ifs_offset[i], s.ifs_enabled[i] = 1, 1.0, 1
            for c in range(3):
                s.ifs_direction[i][c] = d[c]
    s.formula = formula
    a, b = scene.light_from_seed(5)
    keys = dict(keys)
    fog = keys.pop("iter_fog_enabled", 0)
    scene.apply(s, dict(keys, main_light_alfa=a, main_light_beta=b))
    s.iter_fog_enabled = fog
    print(f"[hits] formula {formula} {keys} fog {fog}", flush=True)
    ref, _ = oracle.render(s)
    renderer.set_scene(s)
    for prec in (_abi.PREC_FP64, _abi.PREC_FP32_FIXUP):
        f, st = renderer.render(precision=prec)
        m = compare(f, ref)
        print(f"  {st.hits} hits {m}", flush=True)
        assert st.hits > 0
        assert_parity(m, label=f"precision {prec}")


@pytest.mark.parametrize("w,h", [(3, 2), (67, 41)])
@pytest.mark.parametrize("quality", [1, 2, 8, 9])
def test_fast_ao_items_match_oracle(renderer, quality, w, h):
    """FastAmbientOcclusion2 without estimates (quality 1), as items (2 to 8) and
    as chains (from 9 on), in frames of a few and of several waves' hits."""
    from oracle import oracle
    s = scene.menger_view(w, h, shaded=False)
    a, b = scene.light_from_seed(5)
    scene.apply(s, {"ambient_occlusion_enabled": 1, "fast_ambient_occlusion_mode": 1,
                    "ambient_occlusion_quality": quality, "main_light_alfa": a, "main_light_beta": b})
    print(f"[hits] fast AO quality {quality} {w}x{h}", flush=True)
    ref, _ = oracle.render(s)
    renderer.set_scene(s)
    f64, st = renderer.render(precision=_abi.PREC_FP64)
    m = compare(f64, ref)
    print(f"  {st.hits} hits {m}", flush=True)
    assert st.hits > 0 and m["flips"] == 0 and m["depth_rel_max"] <= 1e-12 and m["psnr_db"] >= 120, m
    assert_planes_exact(m)
    fix, _ = renderer.render(precision=_abi.PREC_FP32_FIXUP)
    assert_parity(compare(fix, ref), label="fixup")


@pytest.mark.parametrize("power", [2.0, 3.0, 7.0, 32.0, 7.5])
def test_fp64_powers_match_oracle(renderer, power):
    """The FP64 Mandelbulb forms r^(p - 1) by products for integer powers from
    2 to 32 and by pow otherwise."""
    from oracle import oracle
    s = scene.mandelbulb_plain(41, 31)
    s.power = power
    print(f"[hits] power {power}", flush=True)
    ref, _ = oracle.render(s)
    renderer.set_scene(s)
    f, st = renderer.render(precision=_abi.PREC_FP64)
    m = compare(f, ref)
    print(f"  {st.hits} hits {m}", flush=True)
    assert st.hits > 0 and m["flips"] == 0
    assert_parity(m, label=f"power {power}")
