"""The renders and image effects that users of this package run, as cases for timing.

Every case goes through the public entry points (Renderer.set_scene,
render_device, render, render_batch, compile_image_device, post_ssao, post_dof,
diff.render) over the sizes of the package's configurations, tests and
benchmark: 96x64 previews to 3840x2160 frames, all four precision modes, and
odd sizes.  A seed sets the light (or the camera), the step jitter and, for the
image effects, the planes.
"""
import math

import numpy as np
import torch

from mandelbulber_amd import Renderer, _abi, diff
from mandelbulber_amd import scene as S

PRECISIONS = {"fp64": _abi.PREC_FP64, "fixup": _abi.PREC_FP32_FIXUP, "march": _abi.PREC_FP32_MARCH,
              "demoivre": _abi.PREC_FP64_DEMOIVRE}

# ---------------------------------------------------------------- the cases


def listed():
    return [
        # a preview thumbnail: launches and the longest ray count, not throughput
        {"name": "preview_96x64_fixup", "kind": "frame", "formula": 2, "power": 8.0, "width": 96, "height": 64,
         "shading": "full", "ao_quality": 4, "precision": "fixup"},
        # the plain method: FP64, no shadow, AO or fog
        {"name": "plain_320x240_fp64", "kind": "frame", "formula": 2, "power": 8.0, "width": 320, "height": 240,
         "shading": "plain", "ao_quality": 4, "precision": "fp64"},
        # the benchmark's frame: hard shadow, AO quality 8, fog
        {"name": "full_1920x1080_fixup", "kind": "frame", "formula": 2, "power": 8.0, "width": 1920,
         "height": 1080, "shading": "full", "ao_quality": 8, "precision": "fixup"},
        # the same shading in the reference's own precision, odd size
        {"name": "full_641x479_fp64", "kind": "frame", "formula": 2, "power": 8.0, "width": 641, "height": 479,
         "shading": "full", "ao_quality": 8, "precision": "fp64"},
        # the folding formulas, shaded, one in each FP32 mode
        {"name": "mandelbox_1280x720_march", "kind": "frame", "formula": 8, "power": 8.0, "width": 1280,
         "height": 720, "shading": "full", "ao_quality": 4, "precision": "march"},
        {"name": "menger_1001x563_fixup", "kind": "frame", "formula": 7, "power": 8.0, "width": 1001,
         "height": 563, "shading": "full", "ao_quality": 4, "precision": "fixup"},
        # a formula of the generic kernels, soft shadow, into host planes (the -nogui path's call)
        {"name": "trig_de_400x300_host", "kind": "host", "formula": 1, "power": 8.0, "width": 400, "height": 300,
         "shading": "soft", "ao_quality": 4, "precision": "fixup"},
        # the largest: a 4K deep zoom into the Mandelbox
        {"name": "deep_zoom_3840x2160_fixup", "kind": "deep", "width": 3840, "height": 2160, "precision": "fixup"},
        # animation: a flight of mixed formulas and resolutions as one graph
        {"name": "flight_12_fixup", "kind": "flight", "frames": 12, "res_div": 1, "precision": "fixup"},
        # inverse rendering: image, MSE, gradient of the nine scene parameters
        {"name": "differentiable_512x512", "kind": "diff", "width": 512, "height": 512},
        # a finished frame to 16 bits with screen-space ambient occlusion
        {"name": "compile_ssao_1920x1080", "kind": "ssao", "width": 1920, "height": 1080, "quality": 20},
        # depth of field of a finished frame
        {"name": "dof_800x600", "kind": "dof", "width": 800, "height": 600, "radius": 10.0},
    ]


def _log_size(rng, lo, hi, aspect):
    """A width log-uniform in [lo, hi] (odd ones among them) and its height."""
    w = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return w, max(16, int(round(w / aspect)) + rng.randrange(2))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "host", "deep", "flight", "diff", "ssao", "dof"])
    aspect = rng.choice([4.0 / 3.0, 16.0 / 9.0, 1.0])
    if kind in ("frame", "host"):
        formula = rng.choice([2, 2, 7, 8]) if kind == "frame" else rng.choice([1, 10, 2, 7, 8])
        precision = rng.choice(["fp64", "fixup", "fixup", "march", "demoivre"])
        # FP64 shades an order slower
        w, h = _log_size(rng, 64, 960 if precision in ("fp64", "demoivre") or kind == "host" else 1920, aspect)
        return {"kind": kind, "formula": formula, "power": rng.choice([8.0, 8.0, round(rng.uniform(6.0, 10.0), 3)]),
                "width": w, "height": h, "shading": rng.choice(["plain", "shadow", "soft", "full"]),
                "ao_quality": rng.randrange(2, 9 if formula == 2 and precision in ("fixup", "march") else 5),
                "precision": precision}
    if kind == "deep":
        w, h = _log_size(rng, 256, 2560, 16.0 / 9.0)
        return {"kind": kind, "width": w, "height": h, "precision": rng.choice(["fixup", "fixup", "fp64"])}
    if kind == "flight":
        return {"kind": kind, "frames": rng.randrange(2, 13), "res_div": rng.choice([1, 2, 3, 5]),
                "precision": "fixup"}
    if kind == "diff":
        w, h = _log_size(rng, 48, 512, 1.0)
        return {"kind": kind, "width": w, "height": min(h, 512)}
    w, h = _log_size(rng, 120, 1920 if kind == "ssao" else 800, aspect)
    if kind == "ssao":
        return {"kind": kind, "width": w, "height": h, "quality": rng.randrange(5, 25)}
    return {"kind": kind, "width": w, "height": h, "radius": round(math.exp(rng.uniform(math.log(4.0), math.log(60.0))), 2)}


# ------------------------------------------------------------------- inputs

_context = {}


def _renderer():
    """The program's one render context."""
    if "r" not in _context:
        _context["r"] = Renderer(0)
    return _context["r"]


def _frame_scene(case, seed):
    w, h, formula, shading = case["width"], case["height"], case["formula"], case["shading"]
    if formula == 7:
        s = S.menger_view(w, h, shaded=False)
    elif formula == 8:
        s = S.mandelbox_view(w, h, shaded=False)
    else:
        s = S.mandelbulb_plain(w, h)
        S.apply(s, {"formula": formula, "power": case["power"]})
    a, b = S.light_from_seed(seed)
    S.apply(s, {"main_light_alfa": a, "main_light_beta": b})
    s.jitter_seed = 1000 + seed % 1000003
    if shading != "plain":
        S.apply(s, {"shadows_enabled": 1, "shadows_cone_angle": 5 if shading == "soft" else 0, "penetrating_lights": 0})
    if shading == "full":
        S.apply(s, {"ambient_occlusion_enabled": 1, "fast_ambient_occlusion_mode": 0,
                    "ambient_occlusion_quality": case["ao_quality"], "volumetric_fog_density": 0.5})
    elif shading == "soft":
        S.apply(s, {"ambient_occlusion_enabled": 1, "fast_ambient_occlusion_mode": 1,
                    "ambient_occlusion_quality": case["ao_quality"]})
    return s


def _deep_scene(case, seed):
    # the benchmark's place, camera and light, the light turned by up to 0.02
    # and another jitter per seed: a shadow ray that grazes the surface at this
    # depth takes 20000 steps, so an arbitrary light takes up to a minute a frame
    s = S.deep_zoom(case["width"], case["height"], seed=1)
    _turn_light(s, np.random.default_rng(seed))
    s.jitter_seed = 1000 + seed % 1000003
    return s


def _turn_light(s, rng):
    s.main_light_alpha += float(rng.uniform(-0.02, 0.02))
    s.main_light_beta += float(rng.uniform(-0.02, 0.02))


def _flight_scenes(case, seed):
    # the benchmark's flight, its lights turned a little and another jitter per seed
    fl = S.flight(case["frames"], seed=0, res_div=case["res_div"])
    rng = np.random.default_rng(seed)
    for s in fl:
        _turn_light(s, rng)
        s.jitter_seed = 1000 + seed % 1000003
    return fl


def _planes(w, h):
    dev = torch.device("cuda:0")
    return {"rgb": torch.empty((3, h, w), dtype=torch.float32, device=dev),
            "z": torch.empty((h, w), dtype=torch.float32, device=dev),
            "colour": torch.empty((3, h, w), dtype=torch.uint8, device=dev),
            "alpha": torch.empty((h, w), dtype=torch.int16, device=dev),
            "opacity": torch.empty((h, w), dtype=torch.int16, device=dev)}


def _finished_frame(w, h, seed):
    """The planes of a finished frame without rendering one: a bumpy ball in
    front of an empty background, depths 2.4 to 3.6 as the Mandelbulb's."""
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:h, 0:w]
    u = (x / w - 0.5) * (w / h) * 2.4 + 0.15 * rng.uniform(-1, 1)
    v = (y / h - 0.5) * 2.4 + 0.15 * rng.uniform(-1, 1)
    bump = np.zeros((h, w))
    for _ in range(6):
        fu, fv, ph = rng.uniform(4, 40), rng.uniform(4, 40), rng.uniform(0, 6.28)
        bump += np.sin(fu * u + fv * v + ph) / 6.0
    rad2 = u * u + v * v
    hit = rad2 < 0.9 + 0.1 * bump
    z = np.where(hit, 3.5 - np.sqrt(np.maximum(1.2 - rad2, 0.0)) + 0.04 * bump, 1e20).astype(np.float32)
    shade = np.clip(0.5 + 0.35 * bump, 0.0, 1.0)
    tint = rng.uniform(0.3, 1.0, 3)
    rgb = np.stack([np.where(hit, shade * t * 1.3, 0.2 * t) for t in tint]).astype(np.float32)
    colour = np.stack([np.where(hit, shade * t * 255, 0) for t in tint]).astype(np.uint8)
    fog = np.clip(0.2 + 0.2 * np.sin(7 * u), 0.0, 1.0)
    opacity = (fog * 65535).astype(np.uint16).view(np.int16)
    alpha = np.where(hit, 65535, fog * 30000).astype(np.uint16).view(np.int16)
    image16 = np.clip(rgb.transpose(1, 2, 0) * 65535, 0, 65535).astype(np.uint16).view(np.int16)
    dev = torch.device("cuda:0")
    t = {"z": z, "rgb": rgb, "colour": colour, "opacity": opacity, "alpha": alpha, "image16": image16}
    return {k: torch.from_numpy(np.ascontiguousarray(a)).to(dev) for k, a in t.items()}


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "r": _renderer(), "precision": PRECISIONS[case.get("precision", "fixup")]}
    if kind == "frame":
        st["scene"] = _frame_scene(case, seed)
        st["planes"] = _planes(case["width"], case["height"])
    elif kind == "host":
        st["scene"] = _frame_scene(case, seed)
    elif kind == "deep":
        st["scene"] = _deep_scene(case, seed)
        st["planes"] = _planes(case["width"], case["height"])
    elif kind == "flight":
        st["scenes"] = _flight_scenes(case, seed)
        st["planes"] = [_planes(s.image_width, s.image_height) for s in st["scenes"]]
    elif kind == "diff":
        st["scene"] = S.differentiable(case["width"], case["height"], seed=100 + seed)
        st["theta"] = torch.tensor(S.get_params(st["scene"]), dtype=torch.float64)
        # the image to match: a smooth one, seeded
        g = torch.Generator().manual_seed(seed)
        c = torch.rand((3, 5, 5), generator=g)
        st["target"] = torch.nn.functional.interpolate(c[None], size=(case["height"], case["width"]), mode="bilinear",
                                                       align_corners=True)[0].to("cuda:0", torch.float64)
    else:
        s = S.mandelbulb_plain(case["width"], case["height"])
        s.jitter_seed = 1000 + seed % 1000003
        st["scene"] = s
        st["frame"] = _finished_frame(case["width"], case["height"], seed)
        st["image16"] = torch.empty_like(st["frame"]["image16"])
        if kind == "ssao":
            s.ssao_quality = case["quality"]
            s.image_gamma, s.contrast, s.brightness = 2.2, 1.1, 1.05
        else:
            s.dof_enabled = 1
            s.dof_radius = case["radius"]
            s.dof_focus = 10.0 * (16.0 + math.log10(2.7))
            st["alpha"] = torch.empty_like(st["frame"]["alpha"])
    return st


# ---------------------------------------------------------------- the calls


def run(st):
    r, kind = st["r"], st["kind"]
    if kind in ("frame", "deep"):
        r.set_scene(st["scene"])
        r.render_device(st["planes"], precision=st["precision"])
        return st["planes"]
    if kind == "host":
        r.set_scene(st["scene"])
        f, _ = r.render(precision=st["precision"])
        return {"rgb": f.rgb, "z": f.z, "colour": f.colour, "alpha": f.alpha.view(np.int16),
                "opacity": f.opacity.view(np.int16)}
    if kind == "flight":
        r.render_batch(st["scenes"], st["planes"], precision=st["precision"])
        return st["planes"]
    if kind == "diff":
        theta = st["theta"].clone().requires_grad_(True)
        img = diff.render(theta, r, st["scene"])
        loss = ((img.double() - st["target"]) ** 2).mean()
        loss.backward()
        return {"image": img.detach(), "loss": loss.detach(), "grad": theta.grad}
    f = st["frame"]
    if kind == "ssao":
        r.compile_image_device(st["scene"], f["rgb"], st["image16"])
        r.post_ssao(st["scene"], f["z"], f["opacity"], [f["colour"][c] for c in range(3)], st["image16"])
        return {"image16": st["image16"]}
    st["image16"].copy_(f["image16"])
    st["alpha"].copy_(f["alpha"])
    r.post_dof(st["scene"], f["z"], st["image16"], st["alpha"])
    return {"image16": st["image16"], "alpha": st["alpha"]}


# ------------------------------------------------------------ the work of it

# floating operations of one formula iteration (additions, products, roots and
# transcendentals counted one each), and iterations of one distance estimate
ITER_FLOPS = {1: 60, 2: 28, 7: 19, 8: 36, 10: 40}
ITERS = {1: 4, 2: 4, 7: 6, 8: 12, 10: 8}
# the part of the frame the object covers, and the estimates of a primary ray,
# of a hit's refinement and normal, of its shadow ray and of one AO direction
HITS = {1: 0.17, 2: 0.17, 7: 0.2, 8: 0.3, 10: 0.2}
STEPS, REFINE, SHADOW, AO = 20, 14, 15, 2


def _render_flops(rays, formula, shading, ao_quality):
    per = ITER_FLOPS[formula] * ITERS[formula] + 12
    hits = rays * HITS[formula]
    calls = rays * STEPS + hits * REFINE
    if shading != "plain":
        calls += hits * SHADOW
    if shading == "full":
        calls += hits * AO * 6.5 * ao_quality * ao_quality
    elif shading == "soft":
        calls += hits * ao_quality * ao_quality
    return calls * per


def work(case):
    kind = case["kind"]
    if kind == "flight":
        sizes = [(s.image_width * s.image_height, s.formula) for s in
                 S.flight(case["frames"], seed=0, res_div=case["res_div"])]
        rays = sum(n for n, _ in sizes)
        return {"bytes": 23 * rays, "flops": sum(_render_flops(n, f, "shadow", 0) for n, f in sizes)}
    rays = case["width"] * case["height"]
    if kind in ("frame", "host"):
        return {"bytes": 23 * rays, "flops": _render_flops(rays, case["formula"], case["shading"], case["ao_quality"])}
    if kind == "deep":
        # every ray hits; the orbit of a point at distance 1e-7 takes about 35 iterations
        return {"bytes": 23 * rays, "flops": rays * (STEPS + REFINE + SHADOW) * (35 * ITER_FLOPS[8] + 12)}
    if kind == "diff":
        # forward as a plain frame with refined hits; backward five estimates with their four tangents per hit,
        # at the hits the forward found
        fwd = _render_flops(rays, 2, "plain", 0)
        return {"bytes": 4 * 3 * rays * 2, "flops": fwd + rays * 0.3 * 5 * 5 * 4 * ITER_FLOPS[2]}
    if kind == "ssao":
        q = case["quality"]
        # rgb, z, colour, opacity in, 16-bit image out; 12 operations per depth sample of the covered half
        return {"bytes": (12 + 4 + 3 + 2 + 6) * rays, "flops": rays * 0.5 * q * (q - 1) * 12}
    # z, image and alpha in, image and alpha out; the blends of each source's disc (radius about 0.2 of the
    # setting in thousandths of the width), 12 operations each
    disc = math.pi * (0.25 * case["radius"] * case["width"] / 1000.0) ** 2
    return {"bytes": (4 + 8 + 8) * rays, "flops": rays * max(1.0, disc) * 12}


# ------------------------------------------------------- depths in 64 bits

def _mix32(x):
    m = 0xFFFFFFFF
    x = (x ^ (x >> 16)) * 0x7FEB352D & m
    x = (x ^ (x >> 15)) * 0x846CA68B & m
    return x ^ (x >> 16)


def _distance(s, p, thr):
    """Distance estimates at the points p (n, 3), by the formulas' definitions."""
    n, dev = p.shape[0], p.device
    out = torch.zeros(n, dtype=torch.float64, device=dev)
    idx = torch.arange(n, device=dev)
    z, c = p.clone(), p
    aux = torch.ones(n, dtype=torch.float64, device=dev)
    for it in range(s.N):
        if s.formula == 2:
            r = z.norm(dim=1)
            th, ph = torch.asin(z[:, 2] / r) * s.power, torch.atan2(z[:, 1], z[:, 0]) * s.power
            rp = r ** (s.power - 1.0)
            aux = rp * aux * s.power + 1.0
            z = torch.stack([th.cos() * ph.cos(), th.cos() * ph.sin(), th.sin()], 1) * (rp * r)[:, None] + c
            r = z.norm(dim=1)
            esc = r > s.bailout
            d = 0.5 * r * r.log() / aux
        elif s.formula == 7:
            z = z.abs().sort(dim=1, descending=True).values * 3.0
            z = z - torch.tensor([2.0, 2.0, 0.0], dtype=torch.float64, device=dev)
            z[:, 2] = torch.where(z[:, 2] > 1.0, z[:, 2] - 2.0, z[:, 2])
            aux = aux * 3.0
            r = z.norm(dim=1)
            esc = r > 1000.0
            d = (r - 2.0) / aux
        else:
            lim, val = s.mb_folding_limit, s.mb_folding_value
            z = torch.where(z > lim, val - z, torch.where(z < -lim, -val - z, z))
            r2 = (z * z).sum(dim=1)
            m2, f2 = s.mb_min_radius ** 2, s.mb_fixed_radius ** 2
            k = torch.where(r2 < m2, torch.full_like(r2, f2 / m2), torch.where(r2 < f2, f2 / r2, torch.ones_like(r2)))
            z = z * k[:, None] * s.mb_scale + c
            aux = aux * k * abs(s.mb_scale) + 1.0
            r = z.norm(dim=1)
            esc = r > 1024.0
            d = r / aux.abs()
        if bool(esc.any()):
            d = d.clamp(min=0.0)
            if it < s.minN:
                d = torch.maximum(d, thr[idx])
            out[idx[esc]] = d[esc]
            keep = ~esc
            idx, z, c, aux = idx[keep], z[keep], c[keep], aux[keep]
            if idx.numel() == 0:
                break
    return out


def _depths(s):
    """Hit depths of the scene's frame (1e20: no hit) by the march of the
    reference's RayMarching with its binary search, in 64 bits."""
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    w, h = s.image_width, s.image_height
    ca, sa, cb, sb, cg, sg = (f(v) for v in (s.alpha, s.beta, s.gamma) for f in (math.cos, math.sin))
    rot = np.array([[ca, -sa, 0], [sa, ca, 0], [0, 0, 1]]) @ np.array([[1, 0, 0], [0, cb, -sb], [0, sb, cb]]) @ \
        np.array([[cg, 0, sg], [0, 1, 0], [-sg, 0, cg]])
    start = torch.from_numpy(np.array(list(s.vp)) - rot @ np.array([0.0, s.zoom / s.persp, 0.0])).to(dev)
    y, x = torch.meshgrid(torch.arange(h, device=dev, dtype=torch.float64),
                          torch.arange(w, device=dev, dtype=torch.float64), indexing="ij")
    v = torch.stack([(x / w - 0.5) * (w / h) * s.persp, torch.ones_like(x), (y / h - 0.5) * s.persp], -1).reshape(-1, 3)
    ray = v @ torch.from_numpy(rot.T.copy()).to(dev)
    n = w * h
    base = _mix32(_mix32(s.jitter_seed ^ 0x9E3779B9) ^ s.frame_no)
    pix = _mix32(torch.arange(n, device=dev, dtype=torch.int64) ^ base)
    kthr = s.persp / w / s.quality
    scan = torch.full((n,), s.view_distance_min, dtype=torch.float64, device=dev)
    step = scan.clone()
    depth = torch.full((n,), 1e20, dtype=torch.float64, device=dev)
    act = torch.arange(n, device=dev)
    hits = [[], [], [], []]
    for i in range(10000):
        if act.numel() == 0:
            break
        sc, thr = scan[act], scan[act] * kthr
        d = _distance(s, start + ray[act] * sc[:, None], thr).clamp(max=3.0)
        hit = d < thr
        for lst, val in zip(hits, (act[hit], d[hit], step[act[hit]], thr[hit])):
            lst.append(val)
        jit = 1.0 - (_mix32(pix[act] ^ i) % 1001).double() / 10000.0 if s.jitter_mode else 1.0
        new = (d - 0.5 * thr) * s.DE_factor * jit
        step[act] = torch.where(hit, step[act], new)
        scan[act] = torch.where(hit, sc, sc + new)
        act = act[~hit & (scan[act] <= s.view_distance_max)]
    idx, d, stp, thr = (torch.cat(lst) for lst in hits)
    t, detail, half = scan[idx].clone(), thr.clone(), stp * 0.5
    live = torch.ones_like(t, dtype=torch.bool)
    low = 1.0 - 0.01 * s.quality
    for _ in range(20):
        live = live & ~((d < thr) & (d > thr * low))
        if not bool(live.any()):
            break
        t = torch.where(live & (d > thr), t + half, torch.where(live & (d < thr * low), t - half, t))
        k = live.nonzero()[:, 0]
        thr[k] = t[k] * kthr
        d[k] = _distance(s, start + ray[idx[k]] * t[k, None], detail[k])
        half = torch.where(live, half * 0.5, half)
    depth[idx] = t
    return depth.reshape(h, w)


def exact(case, seed):
    """The depth plane in 64 bits.  The colours of a frame are a chain of
    shaders over the hits and have no value apart from the renderer's; frames
    of more than 100000 rays, refined hits, the generic formulas, flights and deep
    zooms would take too long."""
    kind = case["kind"]
    if kind in ("frame", "host") and case["formula"] in (2, 7, 8) and case["width"] * case["height"] <= 100000:
        return {"rgb": None, "z": _depths(_frame_scene(case, seed)), "colour": None, "alpha": None, "opacity": None}
    return None
