"""What lm_render promises its callers holds for chunks that take the fused small-chunk kernels as it does for those that
take the kernels per stage."""
import ctypes as C

import pytest
import torch

from landmark_amd import _lib as L
from landmark_amd import scenes

pytestmark = pytest.mark.gpu


def _params(S=128, opt=1, thres=1e-3, gain=6.0, mask=True):
    p = scenes.make_params(seed=7, gridSize=(14, 12, 10), near_far=[0.5, 4.5], n_importance=S, sampling_opt=opt, ndims=3,
                           density_shift=0.0, step_ratio=12.0 / S)
    for t in p.density_plane:
        t.mul_(gain)
    if mask:
        p.alpha_volume = scenes.blob_occupancy((20, 18, 16), 8, 0.5, seed=3)
        p.alpha_aabb = p.aabb.clone()
    p.rayMarch_weight_thres = thres
    return p


def _model(p, **kw):
    from landmark_amd.model import GridNeRFHIP

    return GridNeRFHIP(p, device="cuda", mlp_precision="f16x2", **kw)


def _rays():
    return scenes.pinhole_rays(120, 110, 100.0, scenes.sphere_pose(2.5, 9)).cuda()  # 13200 rays: kernels per stage


def _counts(t):
    return [int(v) & 0xFFFFFFFF for v in t.cpu()]


def test_counter_block_needs_the_alignment_of_its_words_only(gpu_lib):
    """A counter block one word into a buffer (a caller's packed statistics): same counts, same picture, the words around
    it untouched."""
    m = _model(_params())
    rays = _rays()[4000:7000]
    buf = torch.full((L.LM_STAT_WORDS + 2,), 77, dtype=torch.int32, device="cuda")
    odd = buf[1 : 1 + L.LM_STAT_WORDS]
    assert odd.data_ptr() % 8 == 4
    got = []
    for cnt in (torch.zeros(L.LM_STAT_WORDS, dtype=torch.int32, device="cuda"), odd):
        rgb, depth = torch.empty((3000, 3), device="cuda"), torch.empty(3000, device="cuda")
        m.render_into(rays, rgb, depth, counters=cnt)
        torch.cuda.synchronize()
        got.append((rgb, depth, _counts(cnt)))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and got[0][2] == got[1][2]
    assert got[0][2][L.LM_STAT_N_APP] > 1000
    assert int(buf[0]) == 77 and int(buf[-1]) == 77


@pytest.mark.parametrize("S,opt,thres,route", [(128, 1, 1e-4, L.LM_ROUTE_RAYS), (128, 1, 0.0, L.LM_ROUTE_RAYS), (1024, 0, 1e-4, L.LM_ROUTE_RAYS),
                                               (1025, 0, 1e-4, 0), (1300, 0, 0.0, 0), (5000, 0, 1e-3, 0)])
@pytest.mark.parametrize("term", [0.0, 1e-3])
def test_low_thresholds_and_long_rays_in_small_chunks(gpu_lib, S, opt, thres, route, term):
    """Thresholds that let a ray have an entry per sample, and rays the fused kernel does not hold: the same picture and counts as
    the kernels for large chunks give."""
    m = _model(_params(S, opt, thres), term_eps=term)
    rays = _rays()
    whole, _ = m(rays, N_samples=S, chunk=rays.shape[0])
    total = _counts(m.counters)
    n_valid = n_app = at = 0
    for n in (1, 7, 500, 12288, 404):
        st = m._model_struct(S, True)
        assert gpu_lib.lm_render_route(C.byref(st), n) & L.LM_ROUTE_RAYS == route
        part, _ = m(rays[at : at + n], N_samples=S, chunk=n)
        c = _counts(m.counters)
        assert c[L.LM_STAT_OVERFLOW] == 0
        n_valid, n_app = n_valid + c[L.LM_STAT_N_VALID], n_app + c[L.LM_STAT_N_APP]
        assert torch.equal(part["rgb_map"], whole["rgb_map"][at : at + n]) and torch.equal(part["depth_map"], whole["depth_map"][at : at + n])
        at += n
    assert at == rays.shape[0] and n_valid == total[L.LM_STAT_N_VALID] and n_app == total[L.LM_STAT_N_APP] > 1000


@pytest.mark.parametrize("S,opt", [(128, 1), (300, 0), (20, 1)])
def test_rays_by_their_number_of_valid_samples_are_counted(gpu_lib, S, opt):
    """LM_STAT_BINS .. BINS + 3: the same rays per bin, whether a chunk takes the fused kernel or the kernels per stage."""
    m = _model(_params(S, opt))
    rays = _rays()
    cull = m.sample_cull(rays, N_samples=S)
    n = cull["ray_valid"].sum(1)
    assert int(n.max()) >= (64 if S > 64 else 12)
    for at, size in ((0, 13200), (1000, 12200), (5000, 3001), (6000, 5)):
        c = n[at : at + size]
        want = [int(v) for v in ((c >= 64).sum(), ((c >= 32) & (c < 64)).sum(), ((c >= 12) & (c < 32)).sum(), ((c > 0) & (c < 12)).sum())]
        m(rays[at : at + size], N_samples=S, chunk=size)
        got = _counts(m.counters)
        assert got[L.LM_STAT_BINS : L.LM_STAT_BINS + 4] == want and got[L.LM_STAT_N_VALID] == int(c.sum())


@pytest.mark.parametrize("n", [3000, 13200])
def test_a_negative_termination_value_promises_nothing(gpu_lib, n):
    """term_eps below zero is no termination, as zero is; stopping at lost samples is asked for by skip_lost alone."""
    S = 300
    m = _model(_params(S, 0, gain=60.0, mask=False))
    rays = _rays()[:n]
    ws = torch.empty(1 << 30, dtype=torch.uint8, device="cuda")
    marched = {}
    for term, skip in ((0.0, 0), (-1.0, 0), (-1.0, 1), (0.0, 1)):
        st = m._build_model_struct(S, True)
        st.term_eps, st.skip_lost = term, skip
        cnt = torch.zeros(L.LM_STAT_WORDS, dtype=torch.int32, device="cuda")
        rgb, depth = torch.empty((n, 3), device="cuda"), torch.empty(n, device="cuda")
        assert gpu_lib.lm_render_workspace_bytes(C.byref(st), n) <= ws.numel()
        L.check(gpu_lib.lm_render(C.byref(st), rays.data_ptr(), n, ws.data_ptr(), ws.numel(), rgb.data_ptr(), depth.data_ptr(), cnt.data_ptr(),
                                  L.current_stream()), "lm_render")
        torch.cuda.synchronize()
        c = _counts(cnt)
        marched[term, skip] = c[L.LM_STAT_N_VALID] - c[L.LM_STAT_N_MARCHED]
    assert marched[0.0, 0] == 0 and marched[-1.0, 0] == 0
    assert marched[0.0, 1] == marched[-1.0, 1] > 0


def test_colour_sum_of_more_rays_than_one_launch_has_threads_for(gpu_lib):
    """lm_composite_rgb at 2^30 rays and a few: four threads per ray are more than a launch may have."""
    n = (1 << 30) + 37
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 40 GB of device memory")
    cnt, first = torch.zeros(n, dtype=torch.int32, device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
    acc = torch.full((n,), 0.25, device="cuda")
    rgb_map = torch.empty((n, 3), device="cuda")
    w, rgb = torch.tensor([0.5, 0.25], device="cuda"), torch.tensor([[0.25, 0.5, 0.75], [0.5, 0.0, 1.0]], device="cuda")
    at = torch.tensor([0, 1, (1 << 29) - 1, 1 << 29, (1 << 30) - 1, 1 << 30, n - 1], device="cuda")
    cnt[at] = 2
    L.check(gpu_lib.lm_composite_rgb(n, first.data_ptr(), cnt.data_ptr(), w.data_ptr(), rgb.data_ptr(), acc.data_ptr(), 1, rgb_map.data_ptr(),
                                     L.current_stream()), "lm_composite_rgb")
    torch.cuda.synchronize()
    assert torch.equal(rgb_map[at], torch.tensor([[1.0, 1.0, 1.0]], device="cuda").expand(7, 3))
    cnt.zero_()
    cnt[at] = 1
    L.check(gpu_lib.lm_composite_rgb(n, first.data_ptr(), cnt.data_ptr(), w.data_ptr(), rgb.data_ptr(), acc.data_ptr(), 0, rgb_map.data_ptr(),
                                     L.current_stream()), "lm_composite_rgb")
    torch.cuda.synchronize()
    assert torch.equal(rgb_map[at], torch.tensor([[0.125, 0.25, 0.375]], device="cuda").expand(7, 3))
    assert float(rgb_map.sum(dtype=torch.float64)) == 7 * 0.75
