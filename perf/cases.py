"""The work users of the render path have it do, as a list of timed cases.

`listed()` names the cases, `draw(rng)` gives further ones of the same ranges, `prepare(case, seed)` builds what a
program holds before the call (the wrapped model and its inputs, on the GPU), `run(state)` is one pass through the
public entry points, `work(case)` the bytes and operations a pass cannot do without, and `tolerance(case)` how far a
correct implementation of the same precision may differ.

A case is a dict of plain values:
  call    chunk       model(rays): what a server or the reference's fused convention calls per chunk
          loop        renderer_fn(..., exact_chunk=True): the reference's loop with the chunk size the caller insists on
          frame       render_frame(pose): rays, render in chunks, RGBA8 image and depth map
          rows        render_module: the colour network on given features
          density     compute_densityfeature, and
          appearance  compute_appfeature: table lookups at given points
  scene   tiny, multires, production, city, blocks: the scene shapes of landmark_amd.scenes (see `_params`)
  net     arithmetic of the colour network: f32 (the default of the wrapper), f16x2, f16, bf16
"""
import math

import torch

from landmark_amd.model import GridNeRFHIP
from landmark_amd.render import render_frame, renderer_fn
from landmark_amd import scenes

HIDDEN = 128
NET_FLOPS = 2 * (150 * HIDDEN + HIDDEN * HIDDEN + HIDDEN * 3)

# Gathered densities and appearance samples per ray of the scene shapes, over a whole image and over a chunk of pixels
# from its middle, averaged over seeds (work() needs counts that only a render knows).
PER_RAY = {
    "tiny": ((55.0, 12.0), (73.0, 12.5)),
    "multires": ((8.2, 3.4), (15.8, 4.9)),
    "multires_p1": ((8.2, 3.4), (15.8, 4.9)),
    "production": ((73.0, 19.5), (140.0, 28.7)),
    "production_fine": ((294.0, 56.7), (560.0, 83.0)),
    "city": ((11.7, 11.7), (11.7, 11.7)),
    "blocks": ((8.2, 3.4), (16.4, 5.1)),
}


# ---- the cases --------------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: a preview tile of the tiny model with the wrapper's default arithmetic
        {"name": "tile_1k_tiny", "call": "chunk", "scene": "tiny", "net": "f32", "rays": 1024},
        # the reference's default chunk (4096 rays) on the three-orientation multi-resolution model
        {"name": "chunk_4k_multires", "call": "chunk", "scene": "multires", "net": "f16x2", "rays": 4096},
        # a serving chunk of the production shape: one orientation, equal-step sampler at two cells per step (886
        # samples per ray), appearance embedding and density projection
        {"name": "chunk_8k_production", "call": "chunk", "scene": "production", "net": "f16x2", "rays": 8192, "step": 2.0},
        # the reference's own evaluation loop: an image in chunks the caller insists on
        {"name": "loop_540p_4k", "call": "loop", "scene": "multires_p1", "net": "f16x2", "width": 960, "height": 540, "chunk": 4096},
        # a whole small image in one call
        {"name": "image_400_tiny", "call": "chunk", "scene": "tiny", "net": "f32", "rays": 160000},
        # a ragged ray count (no row hint) on a block-stacked model, as dist_render's single-device path calls it
        {"name": "rays_ragged_blocks", "call": "chunk", "scene": "blocks", "net": "f16x2", "rays": 250007},
        # the benchmark's frame: 1080p of the nine-plane model, early termination at the benchmark's value
        {"name": "frame_1080p_multires", "call": "frame", "scene": "multires", "net": "f16x2", "width": 1920, "height": 1080,
         "term_eps": 1e-4 / 6.0},
        # the production shape at the reference's default half a cell per step (3544 samples per ray)
        {"name": "frame_540p_fine_steps", "call": "frame", "scene": "production_fine", "net": "f16x2", "width": 960, "height": 540,
         "step": 0.5},
        # the 4K city block: fp16 tables, 256 samples per ray, fp16 network
        {"name": "frame_4k_city", "call": "frame", "scene": "city", "net": "f16", "width": 3840, "height": 2160, "res": 8192},
        # the colour network alone on 2^23 rows
        {"name": "rows_8m_f16", "call": "rows", "scene": "tiny", "net": "f16", "rows": 1 << 23},
        # table lookups alone: 2^24 random points in three 2048^2 planes of 64 channels
        {"name": "density_16m_64ch", "call": "density", "scene": "tables", "net": "f32", "points": 1 << 24, "res": 2048, "channels": 64},
        # appearance features (lookup and projection) at a ragged number of points of the multi-resolution tables
        {"name": "appearance_1m_multires", "call": "appearance", "scene": "multires", "net": "f16x2", "points": 1000003, "base": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the calls in the proportions of the list, sizes over their whole range."""
    call = rng.choice(["chunk", "chunk", "chunk", "loop", "frame", "frame", "rows", "density", "appearance"])
    if call == "chunk":
        scene = rng.choice(["tiny", "multires", "multires_p1", "production", "blocks"])
        case = {"call": call, "scene": scene, "net": rng.choice(["f32", "f16x2", "f16x2", "bf16"]),
                "rays": _log(rng, 700, 700000 if scene == "production" else 2000000)}
        if scene == "production":
            case["step"] = rng.choice([1.0, 2.0])
    elif call == "loop":
        case = {"call": call, "scene": rng.choice(["multires_p1", "tiny"]), "net": "f16x2", "width": rng.randrange(300, 1280),
                "height": rng.randrange(200, 720), "chunk": _log(rng, 1024, 65536)}
    elif call == "frame":
        scene = rng.choice(["multires", "multires_p1", "production", "city"])
        height = _log(rng, 120, 1080)
        width = 8 * (height * 2 // 9) if rng.random() < 0.7 else height * 16 // 9 + 1  # with and without the row hint
        case = {"call": call, "scene": scene, "net": "f16" if scene == "city" else rng.choice(["f16x2", "f16x2", "f16"]),
                "width": width, "height": height}
        if scene == "city":
            case["res"] = rng.choice([2048, 4096])
        elif scene == "production":
            case["step"] = 2.0
        else:
            case["term_eps"] = rng.choice([0.0, 1e-4 / 6.0])
    elif call == "rows":
        case = {"call": call, "scene": "tiny", "net": rng.choice(["f32", "f16x2", "f16", "bf16"]), "rows": _log(rng, 1000, 1 << 23)}
    elif call == "density":
        case = {"call": call, "scene": "tables", "net": "f32", "points": _log(rng, 4000, 1 << 24), "res": rng.choice([512, 1000, 2048]),
                "channels": rng.choice([16, 32, 64])}
    else:
        case = {"call": call, "scene": "multires", "net": rng.choice(["f32", "f16x2", "f16"]), "points": _log(rng, 4000, 1 << 21),
                "base": rng.choice([256, 512])}
    return case


# ---- scenes -------------------------------------------------------------------------------------
def _params(case, seed):
    """The scene shapes: tables and weights from the seed, occupancy where the shape has it."""
    scene, dev = case["scene"], "cuda"
    if scene == "tiny":  # three 256^2 planes, no occupancy volume, 128 samples per ray
        return scenes.make_params(seed=seed, gridSize=(256, 256, 256), device=dev, near_far=[0.5, 4.5], density_shift=0.0)
    if scene == "tables":  # lookups only
        r, c = case["res"], case["channels"]
        return scenes.make_params(seed=seed, gridSize=(r, r, r), density_n_comp=c, app_n_comp=16, feature_init="uniform", device=dev)
    if scene == "city":  # fp16 tables, flat box, building-like occupancy, 256 samples per ray
        r = case["res"]
        p = scenes.make_params(seed=seed, aabb=((-1, -1, -0.1), (1, 1, 0.1)), gridSize=(r, r, r), device=dev, dtype=torch.float16,
                               near_far=[0.2, 4.0], density_shift=0.0, n_importance=256)
        p.alpha_volume = scenes.heightfield_occupancy((64, 512, 512), 0.15, seed=seed, device=dev)
        p.alpha_aabb = p.aabb.clone()
        return p
    base = case.get("base", 1024)
    cfg = dict(seed=seed, gridSize=(base, base, base), resMode=(1, 2, 4), device=dev, near_far=[0.5, 6.0], density_shift=0.0)
    if scene == "multires":  # three orientations x three levels
        p = scenes.make_params(ndims=3, **cfg)
    elif scene == "multires_p1":  # one orientation
        p = scenes.make_params(ndims=1, **cfg)
    elif scene == "blocks":  # one orientation, 2 x 3 blocks side by side, as merged checkpoints store them
        cfg["gridSize"] = (320, 320, 512)
        p = scenes.make_params(ndims=1, plane_division=(2, 3), **cfg)
    else:  # production, production_fine
        p = scenes.make_params(ndims=1, sampling_opt=0, step_ratio=case["step"], encode_app=True, nonlinear_density=True, **cfg)
        p.basis_den = p.basis_den.abs()
    p.alpha_volume = scenes.blob_occupancy((256, 256, 256), 64, 0.30, seed=seed, device=dev)
    p.alpha_aabb = p.aabb.clone()
    return p


def _pose(case, seed):
    if case["scene"] == "tiny":
        return scenes.sphere_pose(2.5, seed)
    if case["scene"] == "city":
        az, el = 0.05 * (seed % 120), math.radians(30.0)
        eye = (-1.2 * math.cos(el) * math.cos(az), -1.2 * math.cos(el) * math.sin(az), 1.2 * math.sin(el) - 0.1)
        return scenes.look_at_pose(eye, (0.3 * math.cos(az), 0.3 * math.sin(az), -0.1))
    return scenes.orbit_pose(2.6, 1.9, seed % 120)


def _image(case):
    """Width, height and focal length of the image a case renders or takes its rays from."""
    if "width" in case:
        w, h = case["width"], case["height"]
    elif case["scene"] == "tiny":
        w = max(400, math.isqrt(case["rays"] - 1) + 1)
        h = w
    else:
        w, h = 1920, 1080
    focal = 0.5 * w / math.tan(math.radians(25.0)) if case["scene"] == "tiny" else 1483.6378 * (w / 1920.0)
    return w, h, focal


def prepare(case, seed):
    p = _params(case, seed)
    state = {"case": case}
    model = state["model"] = GridNeRFHIP(p, mlp_precision=case["net"], term_eps=case.get("term_eps", 0.0), release_source=True)
    g = torch.Generator(device="cuda").manual_seed(seed)
    call = case["call"]
    if call == "rows":
        state["feat"] = torch.randn((case["rows"], 27), device="cuda", generator=g)
        view = torch.randn((case["rows"], 3), device="cuda", generator=g)
        state["view"] = view / view.norm(dim=1, keepdim=True)
    elif call in ("density", "appearance"):
        state["xyz"] = torch.rand((case["points"], 3), device="cuda", generator=g) * 2 - 1
    else:
        w, h, focal = _image(case)
        state["pose"], state["focal"] = _pose(case, seed), focal
        if model.encode_app:
            state["code"] = seed % 16
        if call != "frame":
            rays = scenes.pinhole_rays(h, w, focal, state["pose"], device="cuda")
            if call == "chunk":  # consecutive pixels from the middle of the image
                n = case["rays"]
                first = (h * w - n) // 2
                rays = rays[first : first + n].clone() if first >= 0 else rays
            state["rays"] = rays
    return state


def run(state):
    case, model = state["case"], state["model"]
    call, code = case["call"], state.get("code")
    if call == "chunk":
        return model(state["rays"], app_code=code)[0]
    if call == "loop":
        return renderer_fn(state["rays"], model, chunk=case["chunk"], app_code=code, exact_chunk=True)[0]
    if call == "frame":
        return render_frame(model, state["pose"], case["height"], case["width"], focal=state["focal"], app_code=code, depth=True)
    if call == "rows":
        return model.render_module(state["view"], state["feat"])
    if call == "density":
        return model.compute_densityfeature(state["xyz"])
    return model.compute_appfeature(state["xyz"])


# ---- what a pass cannot do without ------------------------------------------------------------------
def _planes(case):
    """(texels of one plane, number of planes of that size) per level, and bytes per channel."""
    scene = case["scene"]
    if scene in ("tiny", "tables", "city"):
        r = 256 if scene == "tiny" else case["res"]
        return [(r * r, 3)], 2 if scene == "city" else 4
    if scene == "blocks":
        return [(6 * (320 * r) ** 2, 1) for r in (1, 2, 4)], 4
    base = case.get("base", 1024)
    return [((base * r) ** 2, 3 if scene == "multires" else 1) for r in (1, 2, 4)], 4


def _lookup_bytes(case, n, channels):
    """Texels n random footprints of four touch, each read once."""
    levels, size = _planes(case)
    return sum(k * t * -math.expm1(-4.0 * n / t) * channels * size for t, k in levels)


def work(case):
    levels, _ = _planes(case)
    planes = sum(k for _, k in levels)
    call = case["call"]
    if call == "rows":
        return {"bytes": case["rows"] * 4 * (27 + 3 + 3), "flops": case["rows"] * NET_FLOPS}
    lookup = lambda c: planes * c * 12  # bilinear, linear, product and sum per channel
    if call == "density":
        n, c = case["points"], case["channels"]
        return {"bytes": n * 16 + _lookup_bytes(case, n, c), "flops": n * lookup(c)}
    if call == "appearance":
        n = case["points"]
        return {"bytes": n * (12 + 108) + _lookup_bytes(case, n, 48), "flops": n * (lookup(48) + 2 * planes * 48 * 27)}
    if call == "chunk":
        n_rays = case["rays"]
    else:
        n_rays = case["width"] * case["height"]
    den, app = PER_RAY[case["scene"]][1 if call == "chunk" and n_rays < 300000 else 0]
    if case["scene"] == "production":  # counted at two cells per step
        den, app = den * 2.0 / case["step"], app * 1.4 ** (2.0 / case["step"] - 1.0)
    if case.get("term_eps"):  # a ray stops once next to nothing of it is left
        den = den * 0.69
    n_den, n_app = den * n_rays, app * n_rays
    io = n_rays * (8 if call == "frame" else 24 + 16)
    return {"bytes": int(io + _lookup_bytes(case, n_den, 16) + _lookup_bytes(case, n_app, 48)),
            "flops": int(n_den * lookup(16) + n_app * (lookup(48) + 2 * planes * 48 * 27 + NET_FLOPS))}


def tolerance(case):
    """About four times the largest difference measured: table lookups and the projection against the same sums in
    another order (f32, f16x2) or against 64 bits (16-bit products: 3.0e-4 in fp16, 2.4e-3 in bf16); the colour network
    against 64 bits (5e-8 in f32 and f16x2, 1.9e-5 in fp16, 1.5e-4 in bf16); renders against the f32 network (3e-8,
    7e-6, 5.4e-5).  In a render a weight within rounding of the appearance threshold (1e-3) may fall on the other side:
    such a ray changes by up to the threshold."""
    net, call = case["net"], case["call"]
    if call == "density":
        return {"rel": 1e-5}
    if call == "appearance":
        return {"rel": {"f16": 1.2e-3, "bf16": 1e-2}.get(net, 1e-5)}
    if call == "rows":
        return {"rel": {"f16": 8e-5, "bf16": 6e-4}.get(net, 1e-6)}
    return {"rel": {"f16": 3e-5, "bf16": 2.2e-4}.get(net, 1e-5), "max": 2e-3, "differ": {"f16": 1e-2, "bf16": 1e-2}.get(net, 1e-3)}
