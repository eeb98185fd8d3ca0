"""Density features of many points, put in the order of the tables first, against the kernel that reads the tables per point:
channel counts, ragged sizes, tables whose size no tile divides, planes of several levels, points outside the box and on
its faces, NaN, crowded points (which go to the other kernel), several passes, capture.  Only the order of a sum differs:
K products of magnitude at most |value| summed in fp32, so K * 2^-24 * sum |products| bounds the difference."""
import ctypes as C

import pytest
import torch

from landmark_amd import _lib as L
from landmark_amd import scenes
from landmark_amd.model import GridNeRFHIP

pytestmark = pytest.mark.gpu


def _model(res, channels, levels=(1,), ndims=3, nonlinear=False, seed=3):
    p = scenes.make_params(seed=seed, gridSize=res, density_n_comp=channels, app_n_comp=16, resMode=levels, ndims=ndims, feature_init="uniform",
                           nonlinear_density=nonlinear, device="cuda")
    return GridNeRFHIP(p, mlp_precision="f32")


def _both(m, xyz, ws_bytes=96 << 20):
    arr, n, M = m._plane_array(m._density), len(m._density), xyz.shape[0]
    ref = torch.empty(M, device="cuda")
    got = torch.full((M,), 7e7, device="cuda")
    ws = torch.full((ws_bytes,), 0x7F, dtype=torch.uint8, device="cuda")
    st = L.current_stream()
    L.check(m.lib.lm_gather_density_xyz(arr, n, L.ptr(m._den_w), xyz.data_ptr(), M, ref.data_ptr(), st))
    L.check(m.lib.lm_gather_density_binned(arr, n, L.ptr(m._den_w), xyz.data_ptr(), M, got.data_ptr(), ws.data_ptr(), ws_bytes, st))
    return ref, got


def _points(M, seed=0, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.rand((M, 3), device="cuda", generator=g) * 2 - 1) * scale


def _bound(m):
    # values below 1 in magnitude, products of a plane and a line entry: K * 2^-24 * K
    k = sum(s.C for s in m._density)
    return k * 2.0 ** -24 * k


@pytest.mark.parametrize("res,channels,M", [((40, 56, 24), 16, 4096), ((97, 64, 130), 32, 50001), ((130, 131, 129), 64, 120003), ((512, 300, 70), 64, 400000)])
def test_binned_density_equals_the_direct_lookup(res, channels, M):
    m = _model(res, channels)
    xyz = _points(M)
    xyz[:: 1001] = xyz[:: 1001] * 1.5  # a few outside
    xyz[5] = torch.tensor([1.0, -1.0, 1.0])
    xyz[6] = torch.tensor([-1.0, 1.0, -1.0])
    ref, got = _both(m, xyz)
    assert not torch.equal(ref, got), "the sums run in another order: equal bits mean that the points were not binned"
    assert (ref - got).abs().max().item() <= _bound(m)


def test_levels_and_density_projection():
    m = _model((64, 48, 40), 16, levels=(1, 2, 4), nonlinear=True)
    ref, got = _both(m, _points(100000, seed=1))
    assert (ref - got).abs().max().item() <= _bound(m) and got.min().item() >= 0.0 and got.max().item() > 0.0


def test_a_nan_coordinate_reads_zero_and_touches_nobody_else():
    """A coordinate that is not a number lies outside every table for both kernels: its weights are zero."""
    m = _model((64, 64, 64), 32)
    xyz = _points(60000, seed=2)
    xyz[777] = float("nan")
    ref, got = _both(m, xyz)
    assert ref[777].item() == 0.0 and got[777].item() == 0.0
    assert (ref - got).abs().max().item() <= _bound(m)


@pytest.mark.parametrize("kind", ["cluster", "one point", "plane", "ordered"])
def test_crowded_or_ordered_points_take_the_direct_lookup(kind):
    m = _model((128, 128, 128), 16)
    xyz = _points(100000, seed=4)
    if kind == "cluster":
        xyz = xyz * 0.02
    elif kind == "one point":
        xyz[:] = 0.3
    elif kind == "plane":
        xyz[:, 0] = 0.25
    else:
        xyz = xyz[torch.argsort(torch.floor((xyz[:, 0] + 1) * 64) * 256 + torch.floor((xyz[:, 1] + 1) * 64))].contiguous()
    ref, got = _both(m, xyz)
    assert torch.equal(ref, got)


def test_one_crowded_part_among_spread_points():
    """A fifth of a percent of the points in one texel: below what the sample sees, more than a workgroup's other parts hold"""
    m = _model((256, 256, 256), 64)
    xyz = _points(2000003, seed=5)
    xyz[:: 500] = 0.123
    ref, got = _both(m, xyz, 256 << 20)
    assert (ref - got).abs().max().item() <= _bound(m)


def test_several_passes_and_the_public_entry_point():
    m = _model((48, 48, 48), 16)
    xyz = _points((1 << 24) + 5, seed=6)  # two passes
    ref, got = _both(m, xyz, 512 << 20)
    assert (ref - got).abs().max().item() <= _bound(m)
    del ref, got
    m = _model((512, 512, 512), 64)
    arr, n, M = m._plane_array(m._density), len(m._density), 6500001
    assert m.lib.lm_gather_density_workspace_bytes(arr, n, M) > 0 and m.lib.lm_gather_density_workspace_bytes(arr, n, 100000) == 0
    xyz = _points(M, seed=7)
    ref = torch.empty(M, device="cuda")
    L.check(m.lib.lm_gather_density_xyz(arr, n, None, xyz.data_ptr(), M, ref.data_ptr(), L.current_stream()))
    assert (ref - m.compute_densityfeature(xyz)).abs().max().item() <= _bound(m)


def test_refusals():
    m = _model((48, 48, 48), 16)
    arr, n = m._plane_array(m._density), len(m._density)
    xyz, out, ws = _points(8192), torch.empty(8192, device="cuda"), torch.empty(1024, dtype=torch.uint8, device="cuda")
    st = L.current_stream()
    assert m.lib.lm_gather_density_binned(arr, n, None, xyz.data_ptr(), 8192, out.data_ptr(), ws.data_ptr(), 1024, st) != 0 and b"workspace" in m.lib.lm_last_error()
    assert m.lib.lm_gather_density_binned(arr, n, None, xyz.data_ptr(), 100, out.data_ptr(), ws.data_ptr(), 1024, st) != 0
    assert m.lib.lm_gather_density_binned(arr, n, None, None, 8192, out.data_ptr(), ws.data_ptr(), 1024, st) == -1


def test_capture_and_replay():
    m = _model((96, 96, 96), 32)
    xyz = _points(200000, seed=8)
    arr, n, M = m._plane_array(m._density), len(m._density), xyz.shape[0]
    got = torch.zeros(M, device="cuda")
    ws = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    call = lambda: L.check(m.lib.lm_gather_density_binned(arr, n, None, xyz.data_ptr(), M, got.data_ptr(), ws.data_ptr(), ws.numel(), L.current_stream()))
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for seed in (9, 10, 11):
        xyz.copy_(_points(M, seed=seed))
        graph.replay()
        torch.cuda.synchronize()
        replayed = got.clone()
        got.zero_()
        call()
        torch.cuda.synchronize()
        assert torch.equal(replayed, got)
