"""The marching kernels gather a round's densities with the next plane's loads issued under the present one's arithmetic
(density_sum_rolling).  Same operations in the same order as the lookup per listed sample, so the depth of a render equals
the one formed from lm_density_valid and lm_weights bit for bit (fp32; fp16 up to the order of a sum): full and narrow planes (a lane without channels), one to
nine planes, block-stacked tables, the density projection, both storage types, planes too wide for it, and rays that end
within a round of four."""
import pytest
import torch

from landmark_amd import scenes
from oracle import gridnerf_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dn,ndims,res,opt,fp16,nonlinear,div", [
    (16, 3, (1,), 1, False, False, None), (16, 3, (1, 2, 4), 1, False, False, None), (16, 1, (1,), 0, False, True, None),
    (16, 1, (1, 2, 4), 0, False, True, None), (12, 3, (1,), 1, False, False, None), (4, 1, (1, 2), 0, False, True, None),
    (16, 1, (1, 2), 1, False, False, (2, 3)), (32, 3, (1,), 1, False, False, None), (16, 3, (1, 2), 1, True, False, None),
    (8, 1, (1, 2), 0, True, True, None), (32, 1, (1, 2), 1, True, False, None), (16, 1, (1, 2), 0, True, False, (3, 2)),
])
@pytest.mark.parametrize("n_rays", [14300, 300])
def test_render_depth_equals_the_lookup_per_sample(gpu_lib, dn, ndims, res, opt, fp16, nonlinear, div, n_rays):
    from landmark_amd.model import GridNeRFHIP

    S = 190
    p = scenes.make_params(seed=5, gridSize=(18, 14, 16), near_far=[0.5, 4.5], n_importance=S, sampling_opt=opt, ndims=ndims, resMode=res,
                           density_n_comp=dn, nonlinear_density=nonlinear, plane_division=div, density_shift=0.0, step_ratio=0.3)
    for t in p.density_plane:
        t.mul_(6.0)
    if nonlinear:
        p.basis_den = p.basis_den.abs()
    if div is None:
        p.alpha_volume = scenes.blob_occupancy((20, 18, 16), 8, 0.5, seed=3)
        p.alpha_aabb = p.aabb.clone()
    if fp16:
        p = O.to_fp16_features(p)
    m = GridNeRFHIP(p, device="cuda", mlp_precision="f16x2")
    rays = scenes.pinhole_rays(130, 110, 110.0, scenes.sphere_pose(2.5, 9)).cuda()
    rays = rays if n_rays == rays.shape[0] else rays[7000 : 7000 + n_rays].contiguous()
    out, _ = m(rays, N_samples=S, chunk=rays.shape[0])
    cull = m.sample_cull(rays, N_samples=S)
    w = m.weights(cull, m.density_valid(cull))
    assert w["n_app"] > 50 and (fp16 or m.last_counts()["n_app"] == w["n_app"]) and m.last_counts()["n_valid"] == cull["n_valid"]
    if not fp16:
        assert torch.equal(out["depth_map"], w["depth_map"])
        return
    # The lookup per sample reads eight halves per lane, the march four: K products summed in another order, each sum off by
    # at most K * 2^-24 * sum |products| (below 1 here), times distance scale and path into the opacity, times far into depth
    k = dn * ndims * len(res)
    assert (out["depth_map"] - w["depth_map"]).abs().max().item() <= 4.5 * k * 2.0 ** -24 * p.distance_scale * 4.0


def test_render_does_not_depend_on_the_number_of_workgroups(gpu_lib):
    """fp16 tables of 16 channels march with two workgroups per CU up to a number of rays and with three above it"""
    from landmark_amd.model import GridNeRFHIP

    p = scenes.make_params(seed=6, gridSize=(18, 14, 16), near_far=[0.5, 4.5], n_importance=64, ndims=3, density_shift=0.0)
    for t in p.density_plane:
        t.mul_(6.0)
    m = GridNeRFHIP(O.to_fp16_features(p), device="cuda", mlp_precision="f16")
    limit = 2 * torch.cuda.get_device_properties(0).multi_processor_count * 64 * 4
    rays = scenes.pinhole_rays(400, 400, 380.0, scenes.sphere_pose(2.5, 9)).cuda()[: limit + 65]
    assert rays.shape[0] == limit + 65
    whole, _ = m(rays, chunk=limit + 65)
    for chunk in (limit, limit // 2 + 33):
        parts, _ = m(rays, chunk=chunk)
        assert torch.equal(parts["rgb_map"], whole["rgb_map"]) and torch.equal(parts["depth_map"], whole["depth_map"])
    assert (whole["rgb_map"] != 1.0).any()
