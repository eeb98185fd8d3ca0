"""term_eps = 0 asks for the results of gathering every valid sample.  With finite tables the model lets a ray stop where the
rest cannot change a bit of them: same opacity (through the background), depth, appearance samples and colours, fewer
gathered samples.  Tables holding a NaN or an infinity keep every sample."""
import pytest
import torch

from landmark_amd import _lib as L
from landmark_amd import scenes
from oracle import gridnerf_oracle as O

pytestmark = pytest.mark.gpu


def _scene(gain, opt, S, fp16, thres):
    p = scenes.make_params(seed=5, gridSize=(14, 12, 10), near_far=[0.5, 4.5], n_importance=S, sampling_opt=opt, ndims=3,
                           density_shift=0.0, step_ratio=12.0 / S)
    for t in p.density_plane:
        t.mul_(gain)
    p.rayMarch_weight_thres = thres
    return O.to_fp16_features(p) if fp16 else p


def _render(m, rays, S, chunk):
    out, _ = m(rays, N_samples=S, chunk=chunk)
    torch.cuda.synchronize()
    c = [int(v) & 0xFFFFFFFF for v in m.counters.cpu()]
    return out["rgb_map"].clone(), out["depth_map"].clone(), c[L.LM_STAT_N_VALID], c[L.LM_STAT_N_APP], c[L.LM_STAT_N_MARCHED]


@pytest.mark.parametrize("n", [3000, 20000])  # one kernel from rays to entries, and the kernels per stage
@pytest.mark.parametrize("gain,opt,S,fp16,thres", [(60.0, 1, 128, False, 1e-3), (60.0, 0, 300, False, 1e-3), (400.0, 1, 128, True, 1e-3),
                                                   (60.0, 1, 128, False, 1e-9), (6.0, 1, 64, False, 1e-3)])
def test_stopping_where_the_rest_is_lost_changes_no_bit(gpu_lib, gain, opt, S, fp16, thres, n):
    from landmark_amd.model import GridNeRFHIP

    m = GridNeRFHIP(_scene(gain, opt, S, fp16, thres), device="cuda", mlp_precision="f16x2")
    assert m._finite_densities
    rays = scenes.pinhole_rays(160, 150, 140.0, scenes.sphere_pose(2.5, 9)).cuda()[2000 : 2000 + n]
    got = _render(m, rays, S, n)
    m._finite_densities = False
    m._invalidate()
    want = _render(m, rays, S, n)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and got[2:4] == want[2:4]
    assert want[4] == want[2] and got[4] <= got[2]
    # a small chunk's rays take 64 samples at a time and stop where they have more of them than that
    if gain >= 60.0 and thres == 1e-3 and (n == 20000 or S == 300):
        assert got[4] < got[2]


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf"), 3e38])
def test_tables_that_are_not_finite_keep_every_sample(gpu_lib, value):
    from landmark_amd.model import GridNeRFHIP

    p = _scene(60.0, 1, 128, False, 1e-3)
    p.density_plane[1][0, 3, 5, 6] = value
    m = GridNeRFHIP(p, device="cuda", mlp_precision="f16x2")
    assert not m._finite_densities
    rays = scenes.pinhole_rays(50, 50, 45.0, scenes.sphere_pose(2.5, 9)).cuda()
    got = _render(m, rays, 128, 2500)
    assert got[4] == got[2] > 0


def test_a_model_without_density_tables_can_still_be_asked_for_its_samples(gpu_lib):
    """Sampling, culling, appearance lookups and the colour network need no density tables; a render without them is refused."""
    from landmark_amd.model import GridNeRFHIP

    p = _scene(60.0, 1, 128, False, 1e-3)
    rays = scenes.pinhole_rays(20, 20, 18.0, scenes.sphere_pose(2.5, 9)).cuda()
    want = GridNeRFHIP(p, device="cuda").sample_cull(rays)
    p.density_plane, p.density_line = [], []
    m = GridNeRFHIP(p, device="cuda")
    got = m.sample_cull(rays)
    assert torch.equal(got["ray_valid"], want["ray_valid"]) and got["n_valid"] == want["n_valid"] > 0
    with pytest.raises(L.LandmarkError):
        m(rays)
    p.app_plane, p.app_line = [], []
    with pytest.raises(L.LandmarkError):  # no colour network of width 0
        GridNeRFHIP(p, device="cuda")


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("value,finite", [(1.0, True), (-6e4, True), (float("nan"), False), (-float("inf"), False)])
def test_largest_magnitude_of_the_density_tables_is_found_wherever_it_lies(gpu_lib, fp16, value, finite):
    from landmark_amd.model import GridNeRFHIP

    for table, at in (("density_line", (2, (0, 15, 9, 0))), ("density_plane", (0, (0, 0, 0, 0))), ("density_plane", (2, (0, 15, 8, 6)))):
        p = _scene(6.0, 1, 128, fp16, 1e-3)
        getattr(p, table)[at[0]][at[1]] = value
        assert GridNeRFHIP(p, device="cuda")._finite_densities == finite
