"""Chunks of more than 12288 rays, and small chunks the fused kernel does not hold, go through a kernel per stage: cull and
set-up, march with a quad or a wave per ray, appearance list.  The properties the other files check on a few thousand rays
(which take the fused small-chunk kernels) hold on these routes too."""
import ctypes as C

import pytest
import torch

from landmark_amd import _lib as L
from landmark_amd import scenes
from oracle import gridnerf_oracle as O

pytestmark = pytest.mark.gpu

QUAD, WAVE = "quad per ray", "wave per ray"


def _scene(opt, S, seed=3, mask=True, thres=1e-3, step_ratio=0.3, **kw):
    grid = (9, 11, 13)
    p = scenes.make_params(seed=seed, gridSize=grid, near_far=[0.5, 4.5], n_importance=S, sampling_opt=opt, density_shift=0.0,
                           step_ratio=step_ratio, **kw)
    for t in p.density_plane:
        t.mul_(6.0)
    if mask:
        p.alpha_volume = scenes.blob_occupancy((grid[2], grid[1], grid[0]), 6, 0.45, seed=seed)
        p.alpha_aabb = p.aabb + torch.tensor([[0.01, 0.0, -0.02], [0.0, 0.05, 0.0]])
        p.alpha_mask_filter_thre = 0.0
    p.rayMarch_weight_thres = thres
    return p


def _model(p, **kw):
    from landmark_amd.model import GridNeRFHIP

    return GridNeRFHIP(p, device="cuda", mlp_precision="f16x2", **kw)


def _on_stage_kernels(m, n, S):
    st = m._model_struct(S, True)
    return m.lib.lm_render_route(C.byref(st), n) == 0


def _rays(route):
    if route == QUAD:
        return scenes.pinhole_rays(130, 110, 110.0, scenes.sphere_pose(2.5, 9)).cuda()  # 14300
    return scenes.pinhole_rays(64, 50, 52.0, scenes.sphere_pose(2.5, 9)).cuda()  # 3200


@pytest.mark.parametrize("route,opt,S,thres", [(QUAD, 1, 128, 1e-3), (QUAD, 0, 200, 1e-3), (QUAD, 1, 64, 1e-3), (WAVE, 0, 1100, 1e-4), (WAVE, 0, 4200, 1e-3)])
def test_capacity_overflow_is_reported_and_repeatable(gpu_lib, route, opt, S, thres):
    p = _scene(opt, S, thres=thres, step_ratio=0.3 if S <= 200 else 0.06)
    m = _model(p, capacity="worst")
    rays = _rays(route)
    N = rays.shape[0]
    assert _on_stage_kernels(m, N, S)
    full, _ = m(rays, N_samples=S, chunk=N)
    want = m.last_counts()
    assert want["overflow"] == 0 and want["n_app"] > 1000

    def render(caps):
        st = L.LmModel.from_buffer_copy(m._model_struct(S, True))
        st.cap_valid, st.cap_app = caps
        need = m.lib.lm_render_workspace_bytes(C.byref(st), N)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        rgb, dep = torch.empty((N, 3), device="cuda"), torch.empty((N,), device="cuda")
        cnt = torch.zeros(L.LM_STAT_WORDS, dtype=torch.int32, device="cuda")
        L.check(m.lib.lm_render(C.byref(st), rays.data_ptr(), N, ws.data_ptr(), need, rgb.data_ptr(), dep.data_ptr(), cnt.data_ptr(),
                                L.current_stream()), "lm_render")
        torch.cuda.synchronize()
        c = cnt.cpu().long() & 0xFFFFFFFF
        return rgb, dep, int(c[L.LM_STAT_N_VALID]), int(c[L.LM_STAT_N_APP]), int(c[L.LM_STAT_OVERFLOW])

    rgb, dep, nv, na, over = render((want["n_valid"] // 3, want["n_app"]))
    dropped = ~((rgb == full["rgb_map"]).all(-1) & (dep == full["depth_map"]))
    assert over > 0 and nv == want["n_valid"] and na < want["n_app"]
    assert int(dropped.sum()) <= over and bool((rgb[dropped] == 1.0).all()) and bool((dep[dropped] == 0.0).all())
    rgb, dep, nv, na, over = render((want["n_valid"], want["n_app"] // 2))
    assert over > 0 and nv == want["n_valid"] and na == want["n_app"]
    assert torch.equal(dep, full["depth_map"]) and not torch.equal(rgb, full["rgb_map"])
    rgb, dep, nv, na, over = render((want["n_valid"], want["n_app"]))
    assert over == 0 and torch.equal(rgb, full["rgb_map"]) and torch.equal(dep, full["depth_map"])


@pytest.mark.parametrize("S,width", [(128, 136), (64, 144), (100, 136), (128, 138)])
def test_row_length_hint_changes_nothing(gpu_lib, S, width):
    m = _model(_scene(1, S))
    rays = scenes.pinhole_rays(width, 101, 100.0, scenes.sphere_pose(2.5, 9))[37:].cuda()
    assert _on_stage_kernels(m, rays.shape[0], S)
    a, _ = m(rays, chunk=rays.shape[0])
    m.ray_row_length = width
    b, _ = m(rays, chunk=rays.shape[0])
    assert torch.equal(a["rgb_map"], b["rgb_map"]) and torch.equal(a["depth_map"], b["depth_map"])
    assert float(a["rgb_map"].min()) < 0.99


@pytest.mark.parametrize("route,opt,S,mask,thres", [(QUAD, 1, 128, True, 1e-3), (QUAD, 0, 100, True, 1e-3), (QUAD, 1, 64, False, 1e-3),
                                                    (QUAD, 0, 200, False, 1e-3), (WAVE, 0, 1100, True, 1e-4), (WAVE, 1, 4200, False, 1e-3)])
def test_non_finite_rays_do_not_disturb_their_neighbours(gpu_lib, route, opt, S, mask, thres):
    m = _model(_scene(opt, S, mask=mask, thres=thres, step_ratio=0.3 if S <= 200 else 0.06))
    good = _rays(route)
    N = good.shape[0]
    assert _on_stage_kernels(m, N, S)
    nan, inf = float("nan"), float("inf")
    odd = torch.tensor([
        [nan, 0.0, 0.0, 0.0, 0.0, -1.0], [0.0, 0.0, 2.0, nan, nan, nan], [nan] * 6,
        [inf, 0.0, 0.0, 0.0, 0.0, -1.0], [0.0, 0.0, 2.0, inf, 0.0, -1.0], [0.0, 0.0, -inf, 0.0, 0.0, 1.0],
        [0.0, 0.0, 2.0, 0.0, 0.0, 0.0], [0.1, -0.2, 2.0, 0.0, 0.0, -1.0], [2.0, 0.1, 0.0, -1.0, 0.0, 0.0],
        [0.0, 0.0, 2.0, 0.0, 0.0, -1e30], [1e30, 1e30, 1e30, -1.0, -1.0, -1.0], [0.0, 0.0, 2.0, 1e-30, 0.0, -1e-30],
    ], device="cuda")
    where = torch.arange(odd.shape[0], device="cuda") * (N // 13) + 3
    mixed = good.clone()
    mixed[where] = odd
    keep = torch.ones(N, dtype=torch.bool, device="cuda")
    keep[where] = False
    want, got = m(good, N_samples=S, chunk=N)[0], m(mixed, N_samples=S, chunk=N)[0]
    assert torch.equal(got["rgb_map"][keep], want["rgb_map"][keep]) and torch.equal(got["depth_map"][keep], want["depth_map"][keep])


@pytest.mark.parametrize("opt,S", [(0, 128), (1, 128), (1, 256)])
def test_rays_along_box_faces(gpu_lib, opt, S):
    """Whole words of samples on the boundary of the box test: the depths against the oracle's."""
    p = _scene(opt, S, mask=False, step_ratio=0.05)
    lo, hi = p.aabb[0].tolist(), p.aabb[1].tolist()
    rays = []
    for ax in range(3):
        for face in (lo[ax], hi[ax]):
            f = torch.tensor(face)
            for c in (face, torch.nextafter(f, torch.tensor(10.0)).item(), torch.nextafter(f, torch.tensor(-10.0)).item()):
                for sgn in (1.0, -1.0):
                    o, d = [0.1, -0.2, 1.9], [0.3 * sgn, 0.2, -1.0]
                    if ax == 2:
                        o, d = [-1.7, 0.05, c], [1.0, 0.1 * sgn, 0.0]
                    else:
                        o[ax], d[ax] = c, 0.0
                    rays.append(o + d)
    rays.append([lo[0], lo[1], 1.9, 0.0, 0.0, -1.0])
    rays.append([-1.8, -1.8, 1.8, 1.0, 1.0, -1.0])
    rays = torch.tensor(rays, dtype=torch.float32)
    ref = O.render_chunk(p, rays, N_samples=S, return_aux=True)
    assert ref["ray_valid"].any() and not ref["ray_valid"].all()
    m = _model(p)
    many = rays.repeat(350, 1).cuda()
    assert _on_stage_kernels(m, many.shape[0], S)
    res, _ = m(many, N_samples=S, chunk=many.shape[0])
    got = res["depth_map"].view(350, -1)
    assert torch.equal(got, got[:1].expand_as(got))
    assert (got[0].cpu() - ref["depth_map"]).abs().max().item() <= 1e-4


@pytest.mark.parametrize("route,step,S", [(QUAD, 0.5, -1), (QUAD, 3.0, -1), (WAVE, 0.02, 4200)])
def test_coarse_occupancy_level_changes_nothing(gpu_lib, route, step, S):
    p = scenes.make_params(seed=4, gridSize=(72, 80, 96), near_far=[0.4, 5.0], n_importance=128, sampling_opt=0, step_ratio=step, density_shift=0.0)
    p.alpha_volume = scenes.blob_occupancy((96, 80, 72), 5, 0.06, seed=4)
    p.alpha_aabb = p.aabb + torch.tensor([[0.01, 0.0, -0.02], [0.0, 0.03, 0.0]])
    p.alpha_mask_filter_thre = 0.0
    S = int(p.nSamples) if S < 0 else S
    with_c, without = _model(p), _model(p, coarse_occupancy=False)
    rays = _rays(route)
    N = rays.shape[0]
    assert _on_stage_kernels(with_c, N, S)
    a, b = with_c(rays, N_samples=S, chunk=N)[0], without(rays, N_samples=S, chunk=N)[0]
    assert torch.equal(a["rgb_map"], b["rgb_map"]) and torch.equal(a["depth_map"], b["depth_map"])
    assert with_c.last_counts() == without.last_counts() and with_c.last_counts()["n_valid"] > 1000


@pytest.mark.parametrize("route,S,fp16", [(QUAD, 128, False), (QUAD, 128, True), (WAVE, 4200, False)])
def test_early_termination_bounds(gpu_lib, route, S, fp16):
    """Samples behind a transmittance of 1e-4 weigh less than the appearance threshold: the colour moves by the background's
    share of them, the depth by at most that transmittance times the far end."""
    p = _scene(1, S, resMode=(1, 2))
    if fp16:
        p = O.to_fp16_features(p)
    rays = _rays(route)
    N = rays.shape[0]
    exact, term = _model(p), _model(p, term_eps=1e-4)
    assert _on_stage_kernels(exact, N, S)
    a, b = exact(rays, chunk=N)[0], term(rays, chunk=N)[0]
    assert (a["rgb_map"] - b["rgb_map"]).abs().max().item() <= 1e-4 + 1e-6
    assert (a["depth_map"] - b["depth_map"]).abs().max().item() <= 1e-4 * 4.5 * 1.5
    ca, cb = exact.counters.cpu(), term.counters.cpu()
    assert int(cb[L.LM_STAT_N_MARCHED]) < int(cb[L.LM_STAT_N_VALID]) and int(ca[L.LM_STAT_N_APP]) == int(cb[L.LM_STAT_N_APP])


@pytest.mark.parametrize("route,opt,S,thres", [(QUAD, 1, 128, 1e-3), (QUAD, 0, 100, 1e-3), (WAVE, 0, 1100, 1e-4)])
def test_recorded_into_a_graph(gpu_lib, route, opt, S, thres):
    m = _model(_scene(opt, S, thres=thres, step_ratio=0.3 if S <= 200 else 0.06), capacity="worst")
    shape = (130, 110, 110.0) if route == QUAD else (64, 50, 52.0)
    poses = [scenes.pinhole_rays(*shape, scenes.sphere_pose(2.5, k)).cuda() for k in (9, 3, 14)]
    N = poses[0].shape[0]
    assert _on_stage_kernels(m, N, S)
    st, ws = m._model_struct(S, True), m.workspace(N, S)

    def launch(rays, rgb, depth, cnt):
        L.check(m.lib.lm_render(C.byref(st), rays.data_ptr(), N, ws.data_ptr(), ws.numel(), rgb.data_ptr(), depth.data_ptr(), cnt.data_ptr(),
                                L.current_stream()), "lm_render")

    def eager(rays):
        rgb, depth = torch.full((N, 3), -1.0, device="cuda"), torch.full((N,), -1.0, device="cuda")
        cnt = torch.zeros(L.LM_STAT_WORDS, dtype=torch.int32, device="cuda")
        launch(rays, rgb, depth, cnt)
        torch.cuda.synchronize()
        return rgb, depth, cnt[:8].clone()

    want = [eager(r) for r in poses]
    assert all(int(w[2][L.LM_STAT_N_APP]) > 100 for w in want)
    rays, rgb, depth = poses[0].clone(), torch.empty((N, 3), device="cuda"), torch.empty((N,), device="cuda")
    cnt = torch.zeros(L.LM_STAT_WORDS, dtype=torch.int32, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch(rays, rgb, depth, cnt)
    for k in (0, 1, 2, 0):
        rays.copy_(poses[k])
        rgb.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(rgb, want[k][0]) and torch.equal(depth, want[k][1]) and torch.equal(cnt[:8], want[k][2]), k
        again = eager(poses[(k + 1) % 3])
        assert torch.equal(again[0], want[(k + 1) % 3][0])
