"""Small chunks take one kernel from rays to appearance entries (four rays per workgroup, rounds of 64 samples per ray,
up to 64 words of decisions per ray), larger chunks and longer rays the kernels per stage.  Both walk a ray's samples in
the same order with the same operations, so pictures and counters agree exactly at the sizes where the small-chunk kernel
changes its ways: partly filled workgroups, rays of one word, of a word and a sample, of exactly 64 words and of more, one
and several rounds, one, two and four samples per quad."""
import pytest
import torch

from landmark_amd import scenes
from oracle import gridnerf_oracle as O

pytestmark = pytest.mark.gpu


def _scene(S, opt, fp16=False, dn=16):
    p = scenes.make_params(seed=7, gridSize=(14, 12, 10), near_far=[0.5, 4.5], n_importance=S, sampling_opt=opt, ndims=3,
                           density_n_comp=dn, density_shift=0.0, step_ratio=12.0 / S)
    for t in p.density_plane:
        t.mul_(6.0)
    p.alpha_volume = scenes.blob_occupancy((20, 18, 16), 8, 0.5, seed=3)
    p.alpha_aabb = p.aabb.clone()
    return O.to_fp16_features(p) if fp16 else p


@pytest.mark.parametrize("S,opt,fp16,dn,term", [(1, 1, False, 16, 0.0), (63, 1, False, 16, 0.0), (65, 0, False, 16, 1e-3), (128, 1, True, 16, 0.0),
                                                (200, 0, False, 32, 0.0), (4096, 0, False, 16, 0.0), (4097, 0, False, 16, 1e-3)])
def test_small_chunk_kernel_equals_the_stage_kernels(gpu_lib, S, opt, fp16, dn, term):
    from landmark_amd.model import GridNeRFHIP

    m = GridNeRFHIP(_scene(S, opt, fp16, dn), device="cuda", mlp_precision="f16x2", term_eps=term)
    rays = scenes.pinhole_rays(120, 110, 100.0, scenes.sphere_pose(2.5, 9)).cuda()  # 13200 rays: kernels per stage
    whole, _ = m(rays, N_samples=S, chunk=rays.shape[0])
    total = m.last_counts()
    assert total["overflow"] == 0 and (S < 63 or total["n_app"] > 1000)
    n_valid = n_app = at = 0
    for n in (1, 3, 4, 5, 64, 131, 1000, 5000, 6992):
        part, _ = m(rays[at : at + n], N_samples=S, chunk=n)
        c = m.last_counts()
        n_valid, n_app = n_valid + c["n_valid"], n_app + c["n_app"]
        assert torch.equal(part["rgb_map"], whole["rgb_map"][at : at + n]) and torch.equal(part["depth_map"], whole["depth_map"][at : at + n])
        at += n
    assert at == rays.shape[0] and n_valid == total["n_valid"] and n_app == total["n_app"]
