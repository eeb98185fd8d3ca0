"""The marching kernels gather a round's densities with the next plane's loads issued under the present one's arithmetic
(density_sum_rolling).  Same operations in the same order as the lookup per listed sample, so the depth of a render equals
the one formed from lm_density_valid and lm_weights bit for bit: full and narrow planes (a lane without channels), one to
nine planes, block-stacked tables, the density projection, both storage types, planes too wide for it, tables whose 32-bit offsets
pass 2^31, tables of 4 GB (which keep the plain form and 64-bit offsets), and rays that end within a round of four.  fp16 tables of up to
16 channels are marched four channels to a lane and looked up per sample eight to a lane; their render equals that of the same
values in fp32 tables, which are read four to a lane everywhere."""
import copy

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
    _check(p, S, n_rays)


def _check(p, S, n_rays):
    from landmark_amd.model import GridNeRFHIP

    m = GridNeRFHIP(p, device="cuda", mlp_precision="f16x2")
    rays = scenes.pinhole_rays(130, 110, 110.0, scenes.sphere_pose(2.5, 9)).cuda()
    rays = rays if n_rays == rays.shape[0] else rays[7000 : 7000 + n_rays].contiguous()
    out, _ = m(rays, N_samples=S, chunk=rays.shape[0])
    counts = m.last_counts()
    if p.density_plane[0].dtype == torch.float16 and p.density_plane[0].shape[1] <= 16:
        q = copy.copy(p)
        for name in ("density_plane", "density_line", "app_plane", "app_line"):
            setattr(q, name, [t.float() for t in getattr(p, name)])
        m = GridNeRFHIP(q, device="cuda", mlp_precision="f16x2")
    cull = m.sample_cull(rays, N_samples=S)
    w = m.weights(cull, m.density_valid(cull))
    assert w["n_app"] > 50 and counts["n_app"] == w["n_app"] and counts["n_valid"] == cull["n_valid"]
    assert torch.equal(out["depth_map"], w["depth_map"]) and out["depth_map"].unique().numel() > 50


@pytest.mark.parametrize("size,fp16,nonlinear", [
    ((8192, 8191), False, False),  # offsets up to 2^32 - 2^19
    ((8192, 8192), False, False), ((8192, 8192), False, True), ((16384, 8192), True, False)])  # 2^32 bytes: the plain form
@pytest.mark.parametrize("n_rays", [14300, 300])
def test_tables_of_up_to_4_gb_and_beyond(gpu_lib, size, fp16, nonlinear, n_rays):
    p = scenes.make_params(seed=8, gridSize=(*size, 16), near_far=[0.5, 4.5], n_importance=64, ndims=1, nonlinear_density=nonlinear,
                           density_n_comp=16, app_n_comp=16, density_shift=0.0, device="cuda", dtype=torch.float16 if fp16 else torch.float32)
    for t in p.density_plane:
        t.mul_(6.0)
    if nonlinear:
        p.basis_den = p.basis_den.abs()
    _check(p, 64, n_rays)


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
