"""The back half of a render has two forms: one kernel per stage (large chunks) and one kernel from appearance entries to
colours (small chunks).  Both do the same operations in the same order, so pictures agree exactly, in every arithmetic mode
and for every channel width, storage type and number of planes the small form covers; widths and mixtures it does not cover
take the kernels per stage.  compute_appfeature has both forms too (few and many points), and
a third one through memory for what they do not cover."""
import pytest
import torch

from landmark_amd import scenes
from oracle import gridnerf_oracle as O

pytestmark = pytest.mark.gpu


def _scene(an, ndims, res=(1,), fp16=False, seed=7):
    p = scenes.make_params(seed=seed, gridSize=(14, 12, 10), resMode=res, near_far=[0.5, 4.5], ndims=ndims, density_n_comp=16,
                           app_n_comp=an, density_shift=0.0, n_importance=64)
    for t in p.density_plane:
        t.mul_(6.0)
    return O.to_fp16_features(p) if fp16 else p


@pytest.mark.parametrize("net", ["f32", "f16x2", "f16", "bf16"])
@pytest.mark.parametrize("an,ndims,res,fp16", [(16, 1, (1,), False), (32, 3, (1,), False), (48, 3, (1, 2, 4), False), (64, 3, (1, 2), False),
                                               (16, 3, (1,), True), (32, 1, (1, 2), True), (48, 3, (1,), True), (64, 3, (1,), True)])
def test_small_chunk_shading_equals_the_stage_kernels(gpu_lib, net, an, ndims, res, fp16):
    from landmark_amd.model import GridNeRFHIP

    m = GridNeRFHIP(_scene(an, ndims, res, fp16), device="cuda", mlp_precision=net)
    rays = scenes.pinhole_rays(120, 110, 100.0, scenes.sphere_pose(2.5, 9)).cuda()  # 13200 rays: kernels per stage
    whole, _ = m(rays, chunk=rays.shape[0])
    assert m.last_counts()["n_app"] > 1000 and (whole["rgb_map"] < 0.99).any()
    at = 6000  # the middle of the picture
    for n in (1, 2, 31, 500, 4096):  # fewer and more than 32 entries, many tiles per workgroup
        part, _ = m(rays[at : at + n], chunk=n)
        assert torch.equal(part["rgb_map"], whole["rgb_map"][at : at + n])
        assert torch.equal(part["depth_map"], whole["depth_map"][at : at + n])


@pytest.mark.parametrize("net", ["f32", "f16x2", "f16", "bf16"])
@pytest.mark.parametrize("an,ndims,res,fp16", [(16, 1, (1,), False), (32, 3, (1, 2), False), (48, 3, (1,), False), (64, 3, (1,), False),
                                               (64, 3, (1, 2, 3, 4), False),  # basis_mat too large for LDS in the wide modes
                                               (16, 3, (1,), True), (32, 1, (1,), True), (48, 3, (1, 2), True), (64, 1, (1,), True)])
def test_appearance_features_of_points_equal_products_and_projection(gpu_lib, net, an, ndims, res, fp16):
    from landmark_amd.model import GridNeRFHIP

    m = GridNeRFHIP(_scene(an, ndims, res, fp16), device="cuda", mlp_precision=net)
    g = torch.Generator().manual_seed(3)
    for n in (1, 31, 32, 33, 5000, 99001):  # a tile per workgroup, several of them, a tile per wave
        xyz = torch.rand((n, 3), generator=g) * 2.6 - 1.3  # some outside the tables
        xyz[0] = float("nan")
        got = m.compute_appfeature(xyz)
        assert got.shape == (n, 27)
        assert torch.equal(got, m.basis(m.app_products(xyz)))
    assert m.compute_appfeature(torch.zeros((0, 3))).shape == (0, 27)
