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
