"""Density features of many points, put in the order of the tables first: against sums in 64 bits and against the kernel that
reads the tables per point.  Channel counts, ragged sizes, tables whose size no tile divides, planes of several levels, points
outside the box and on its faces, NaN, points that crowd in some blocks (several units to a block, several groups to a column),
few points per texel, crowded points (which go to the other kernel), several passes, capture.

The reference takes the kernels' fp32 weights and adds in 64 bits.  A product of a texel's share and a line entry passes at most
2 + 3 roundings on the plane, 2 on the line, 1 or 2 in the product, and its channel's sum at most 4 in a lane, 4 between lanes, one
per plane: 17 + planes, each 2^-24 of the sum of magnitudes.  The lookup per point adds a lane's channels of all planes in one
chain, K / 4 long."""
import ctypes as C

import numpy as np
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


def _axis(c, size):
    """First corner (clamped as the kernels do) and the weights of both corners along an axis, fp32"""
    i = ((c + 1.0) / 2.0) * float(size - 1)
    f = torch.floor(i)
    w1, w0 = i - f, (f + 1.0) - i
    n = torch.nan_to_num(f, nan=-2.0).clamp(-2.0, float(size)).long()
    inside = lambda k: (k >= 0) & (k < size)
    return n.clamp(0, size - 1), (n + 1).clamp(0, size - 1), torch.where(inside(n), w0, 0.0), torch.where(inside(n + 1), w1, 0.0)


def _in_64_bits(m, xyz):
    """(sums, sums of magnitudes) of every point"""
    p, total, mags = m.p, [], []
    for q in xyz.split(1 << 17):
        s, a = torch.zeros(len(q), dtype=torch.float64, device="cuda"), torch.zeros(len(q), dtype=torch.float64, device="cuda")
        col = 0
        for k, pl in enumerate(m._density):
            x0, x1, wx0, wx1 = _axis(q[:, pl.ax0], pl.W)
            y0, y1, wy0, wy1 = _axis(q[:, pl.ax1], pl.H)
            l0, l1, wl0, wl1 = _axis(q[:, pl.axl], pl.Len)
            plane, line = p.density_plane[k][0].cuda(), p.density_line[k][0, :, :, 0].cuda()  # [C, H, W], [C, Len]
            v = va = 0.0
            for y, wy in ((y0, wy0), (y1, wy1)):
                for x, wx in ((x0, wx0), (x1, wx1)):
                    t = plane[:, y, x].double() * (wx * wy).double()
                    v, va = v + t, va + t.abs()
            ln = [line[:, i].double() * w.double() for i, w in ((l0, wl0), (l1, wl1))]
            w = 1.0 if p.basis_den is None else p.basis_den.reshape(-1)[col : col + pl.C].cuda().double()[:, None]
            s += (v * (ln[0] + ln[1]) * w).sum(0)
            a += (va * (ln[0].abs() + ln[1].abs()) * (w if isinstance(w, float) else w.abs())).sum(0)
            col += pl.C
        total.append(s if p.basis_den is None else s.clamp(min=0.0))
        mags.append(a)
    return torch.cat(total), torch.cat(mags)


def _check(m, xyz, ref, got, sorts=True):
    """Both results within their bounds of the sums in 64 bits; the points did take the sorted path"""
    if sorts:
        assert not torch.equal(ref, got), "the sums run in another order: equal bits mean that the points were not sorted"
    want, mags = _in_64_bits(m, xyz)
    planes, K = len(m._density), sum(s.C for s in m._density)
    assert ((got.double() - want).abs() <= (17 + planes) * 2.0 ** -24 * mags).all()
    assert ((ref.double() - want).abs() <= (17 + K // 4) * 2.0 ** -24 * mags).all()


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


@pytest.mark.parametrize("res,channels,M", [((40, 56, 24), 16, 4096), ((97, 64, 130), 32, 50001), ((130, 131, 129), 64, 120003), ((512, 300, 70), 64, 400000)])
def test_binned_density_equals_the_direct_lookup(res, channels, M):
    m = _model(res, channels)
    xyz = _points(M)
    xyz[:: 1001] = xyz[:: 1001] * 1.5  # a few outside
    xyz[5] = torch.tensor([1.0, -1.0, 1.0])
    xyz[6] = torch.tensor([-1.0, 1.0, -1.0])
    ref, got = _both(m, xyz)
    _check(m, xyz, ref, got)


def test_levels_and_density_projection():
    m = _model((64, 48, 40), 16, levels=(1, 2, 4), nonlinear=True)
    xyz = _points(100000, seed=1)
    ref, got = _both(m, xyz)
    _check(m, xyz, ref, got)
    assert got.min().item() >= 0.0 and got.max().item() > 0.0


def test_a_nan_coordinate_reads_zero_and_touches_nobody_else():
    """A coordinate that is not a number lies outside every table for both kernels: its weights are zero."""
    m = _model((64, 64, 64), 32)
    xyz = _points(60000, seed=2)
    xyz[777] = float("nan")
    ref, got = _both(m, xyz)
    assert ref[777].item() == 0.0 and got[777].item() == 0.0
    _check(m, xyz, ref, got)


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


def _replay(xyz):
    """What k_bin_decide and k_bin_scan see, on the host: (largest share of a part of a plane in the sample, points of the fullest
    block, units of the fullest column)"""
    x, M, side = xyz.cpu().numpy(), len(xyz), 1
    while side < 12 and side ** 3 * 10000 < M:
        side += 1
    strip = lambda c, n: np.clip((c + np.float32(1)) * np.float32(0.5 * n), 0, n - 1).astype(np.int64)
    n = np.bincount((strip(x[:, 0], side) * side + strip(x[:, 1], side)) * side + strip(x[:, 2], side), minlength=side ** 3)
    units = ((n + 16383) // 16384).reshape(side, side, side)
    k, stride = np.arange(4096), M // 4096
    q = x[np.minimum(k * stride + (k * 2654435761 % 2 ** 32 >> 8) % stride, M - 2)]
    most = max(np.bincount(strip(q[:, a], 64) * 64 + strip(q[:, b], 64)).max() for a, b in ((0, 1), (0, 2), (1, 2)))
    return int(most), int(n.max()), int(max(units.sum(a).max() for a in range(3)))


@pytest.mark.parametrize("M,share,channels", [(300001, 0.4, 32), (2000003, 0.36, 16)])
def test_blocks_of_several_units_and_columns_of_several_groups(M, share, channels):
    """Half of the points in the middle `share` of every axis: spread enough to be sorted, but blocks hold several times the
    average, so that they become several units (and, of the larger number, a column more than one group of 16)."""
    m = _model((96, 120, 110), channels)
    xyz = _points(M, seed=5)
    xyz[::2] *= share
    most, block, column = _replay(xyz)
    assert most <= 16 and block > 16384 and (M < 2000000 or column > 16)
    ref, got = _both(m, xyz, 256 << 20)
    _check(m, xyz, ref, got)


@pytest.mark.parametrize("M", [20000, 60000, 90000, 140000])
def test_few_points_per_texel(M):
    """Sub-tiles with fewer points than half their texels are not staged, their points read the table: none, some and most"""
    m = _model((512, 300, 400), 32)
    xyz = _points(M, seed=12)
    ref, got = _both(m, xyz)
    _check(m, xyz, ref, got)


def test_one_crowded_texel_among_spread_points():
    """A tenth of a percent of the points in one texel: below what the sample sees, more than a sub-tile's other points"""
    m = _model((256, 256, 256), 64)
    xyz = _points(2000003, seed=5)
    xyz[:: 1000] = 0.123
    assert _replay(xyz)[0] <= 16
    ref, got = _both(m, xyz, 256 << 20)
    _check(m, xyz, ref, got)


def test_several_passes_and_the_public_entry_point():
    m = _model((48, 48, 48), 16)
    xyz = _points((1 << 24) + 5, seed=6)  # two passes
    ref, got = _both(m, xyz, 512 << 20)
    _check(m, xyz, ref, got)
    assert not torch.equal(ref[: 1 << 23], got[: 1 << 23]) and not torch.equal(ref[1 << 24 :], got[1 << 24 :])  # in both passes
    del ref, got
    m = _model((512, 512, 512), 64)
    arr, n, M = m._plane_array(m._density), len(m._density), 6500001
    assert m.lib.lm_gather_density_workspace_bytes(arr, n, M) > 0 and m.lib.lm_gather_density_workspace_bytes(arr, n, 100000) == 0
    xyz = _points(M, seed=7)
    ref = torch.empty(M, device="cuda")
    L.check(m.lib.lm_gather_density_xyz(arr, n, None, xyz.data_ptr(), M, ref.data_ptr(), L.current_stream()))
    _check(m, xyz, ref, m.compute_densityfeature(xyz))


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
