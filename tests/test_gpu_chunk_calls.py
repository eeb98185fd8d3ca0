"""lm_render_chunks: many chunks in one call of the library, on one to five streams, give what one render of all rays gives,
with a counter block per chunk; full and ragged last chunks, a single chunk, chunks whose workspace overflows (repeated)."""
import ctypes as C

import pytest
import torch

from landmark_amd import _lib as L
from landmark_amd import scenes

pytestmark = pytest.mark.gpu


def _model(**kw):
    from landmark_amd.model import GridNeRFHIP

    p = scenes.make_params(seed=7, gridSize=(14, 12, 10), near_far=[0.5, 4.5], n_importance=64, ndims=3, density_shift=0.0)
    for t in p.density_plane:
        t.mul_(6.0)
    return GridNeRFHIP(p, device="cuda", mlp_precision="f16x2", **kw)


def _rays(n):
    return scenes.pinhole_rays(130, 110, 110.0, scenes.sphere_pose(2.5, 9)).cuda()[:n].contiguous()


@pytest.mark.parametrize("n,step", [(14300, 1024), (14300, 1430), (13000, 13000), (100, 1), (12289, 12288), (5, 1000)])
@pytest.mark.parametrize("streams", [1, 4, 5])
def test_chunks_of_one_call_equal_one_render(gpu_lib, n, step, streams):
    m = _model()
    rays = _rays(n)
    whole, _ = m(rays, chunk=n, streams=1)
    got, _ = m(rays, chunk=step, streams=streams)
    assert torch.equal(got["rgb_map"], whole["rgb_map"]) and torch.equal(got["depth_map"], whole["depth_map"])
    assert n < 1000 or (whole["rgb_map"] != 1.0).any()


def test_overflowing_chunks_are_repeated(gpu_lib):
    rays = _rays(14300)
    want, _ = _model(capacity="worst")(rays, chunk=14300)
    m = _model()
    m.small_workspace, m.samples_per_ray = 0, [4.0, 0.5]
    got, _ = m(rays, chunk=5000, streams=3)
    assert torch.equal(got["rgb_map"], want["rgb_map"]) and torch.equal(got["depth_map"], want["depth_map"])
    assert m.samples_per_ray[0] > 4.0


def test_counter_blocks_and_refusals(gpu_lib):
    m = _model()
    rays, step, n = _rays(14300), 4000, 14300
    m(rays, chunk=n)
    total = m.last_counts()
    st = m._model_struct(64, True)
    ws = torch.empty(m.lib.lm_render_workspace_bytes(C.byref(st), step), dtype=torch.uint8, device="cuda")
    rgb, dep = torch.empty((n, 3), device="cuda"), torch.empty((n,), device="cuda")
    cnt = torch.zeros((4, L.LM_STAT_WORDS), dtype=torch.int32, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream

    def call(k, size, step=step):
        return m.lib.lm_render_chunks(C.byref(st), rays.data_ptr(), n, step, k, (C.c_void_p * 1)(stream), (C.c_void_p * 1)(ws.data_ptr()),
                                      (C.c_size_t * 1)(size), rgb.data_ptr(), dep.data_ptr(), cnt.data_ptr())

    assert call(1, ws.numel()) == 0
    host = cnt.cpu().long() & 0xFFFFFFFF
    assert host[:, L.LM_STAT_N_VALID].sum() == total["n_valid"] and host[:, L.LM_STAT_N_APP].sum() == total["n_app"]
    assert call(0, ws.numel()) == -1 and call(1, ws.numel(), 0) == -1
    assert call(1, 1024) != 0 and b"workspace" in m.lib.lm_last_error()
