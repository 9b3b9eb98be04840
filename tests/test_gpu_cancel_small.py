"""mbr_cancel on frames whose rays all fit the GPU at once: the march's waves
take them by number, without an add to the shared queue, and a cancel made
before the render still leaves every ray empty (the reference's programClosed
test comes before every pixel, src/Render3D.cpp:369-378)."""
import numpy as np
import pytest

from mandelbulber_amd import _abi, scene
from mandelbulber_amd._lib import MbrError

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


def _planes(w, h):
    import torch
    d = torch.device("cuda:0")
    planes = {"rgb": torch.zeros((3, h, w), device=d), "z": torch.zeros((h, w), device=d),
              "colour": torch.full((3, h, w), 7, dtype=torch.uint8, device=d),
              "alpha": torch.zeros((h, w), dtype=torch.int16, device=d),
              "opacity": torch.zeros((h, w), dtype=torch.int16, device=d)}
    torch.cuda.synchronize()  # the context renders on a stream of its own
    return planes


@pytest.mark.parametrize("call", ["render_device", "render_device_noalloc"])
@pytest.mark.parametrize("formula,prec", [(2, _abi.PREC_FP64), (2, _abi.PREC_FP32_FIXUP), (2, _abi.PREC_FP32_MARCH),
                                          (13, _abi.PREC_FP64)])
@pytest.mark.parametrize("w,h", [(9, 7), (160, 120)])
def test_cancelled_small_frame_is_empty(renderer, w, h, formula, prec, call):
    s = scene.mandelbulb_full(w, h, seed=1)
    s.ao_quality = 2
    if formula == 13:
        s.formula, s.power, s.N = 13, 2.0, 20
    renderer.set_scene(s)
    render = getattr(renderer, call)
    print(f"[cancel] {call} {w}x{h} formula {formula} precision {prec}", flush=True)
    want = _planes(w, h)
    assert render(want, precision=prec).hits > 0
    renderer.cancel()
    got = _planes(w, h)
    with pytest.raises(MbrError) as e:
        render(got, precision=prec)
    assert e.value.rc == -6
    assert bool((got["z"] > 1e19).all()) and not bool(got["colour"].any())
    again = _planes(w, h)
    render(again, precision=prec)
    assert all(np.array_equal(want[k].cpu().numpy(), again[k].cpu().numpy(), equal_nan=True) for k in want)
