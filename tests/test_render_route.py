"""Which kernels a chunk takes follows from its rays, samples per ray, appearance threshold and channel widths; asked on the
host, nothing is launched."""
import ctypes as C

import pytest

from landmark_amd import _lib as L


def _host_model(S, thres, app_channels=48, prec=L.LM_MLP_F16X2):
    m = L.LmModel()
    m.geom.S, m.geom.sampler = S, L.LM_SAMPLER_HULL
    m.geom.tab_a = m.geom.tab_t = 16
    m.n_planes = 3
    for k in range(3):
        for arr, c in ((m.density, 16), (m.app, app_channels)):
            arr[k].plane = arr[k].line = 16
            arr[k].H = arr[k].W = arr[k].Len = 8
            arr[k].C = c
    m.mlp_prec, m.weight_thres = prec, thres
    return m


@pytest.fixture(scope="module")
def lib():
    import os

    if not os.path.exists(L.SO_PATH):
        from landmark_amd import build

        build.build(verbose=False)
    return L.load()


@pytest.mark.parametrize("S,thres,n,fused", [
    (128, 1e-3, 4096, True), (128, 1e-4, 4096, True), (128, 0.0, 4096, True), (128, -1.0, 4096, True),  # a slot per sample
    (1024, 1e-9, 4096, True), (1025, 1e-9, 100, False), (1025, 1e-3, 100, True), (1025, 1e-4, 100, False), (1025, 0.0, 100, False),
    (4096, 1e-3, 4096, True), (4097, 1e-3, 4096, False), (128, 1e-3, 12288, True), (128, 1e-3, 12289, False), (128, float("nan"), 100, True),
    (2048, float("nan"), 100, False)])
def test_small_chunks_take_one_kernel_where_their_entries_fit(lib, S, thres, n, fused):
    got = lib.lm_render_route(C.byref(_host_model(S, thres)), n)
    assert got >= 0 and bool(got & L.LM_ROUTE_RAYS) == fused
    if not fused:
        assert got == 0


@pytest.mark.parametrize("prec,S,n,fused", [(L.LM_MLP_F16X2, 128, 12288, True), (L.LM_MLP_F16X2, 384, 8192, True), (L.LM_MLP_F16X2, 385, 8192, False),
                                            (L.LM_MLP_F32, 128, 4096, True), (L.LM_MLP_F32, 128, 4097, False), (L.LM_MLP_F32, 1024, 1024, False)])
def test_shading_in_one_kernel_up_to_a_number_of_candidate_samples(lib, prec, S, n, fused):
    got = lib.lm_render_route(C.byref(_host_model(S, 1e-3, prec=prec)), n)
    assert got == L.LM_ROUTE_RAYS | (L.LM_ROUTE_SHADE if fused else 0)
    assert lib.lm_render_route(C.byref(_host_model(S, 1e-3, app_channels=40, prec=prec)), n) == L.LM_ROUTE_RAYS


@pytest.mark.parametrize("prec,thres,n,fused", [(L.LM_MLP_F16X2, 0.0, 8192, True), (L.LM_MLP_F16X2, 0.0, 8193, False), (L.LM_MLP_F16X2, 7e-5, 8193, False),
                                                (L.LM_MLP_F16X2, 1e-4, 8193, True), (L.LM_MLP_F16X2, -1.0, 8193, False), (L.LM_MLP_F32, 0.0, 1365, True),
                                                (L.LM_MLP_F32, 0.0, 1366, False), (L.LM_MLP_F32, 1e-4, 1366, True)])
def test_shading_limit_where_nearly_every_valid_sample_is_an_entry(lib, prec, thres, n, fused):
    got = lib.lm_render_route(C.byref(_host_model(128, thres, prec=prec)), n)
    assert got == L.LM_ROUTE_RAYS | (L.LM_ROUTE_SHADE if fused else 0)


def test_bad_arguments_are_refused(lib):
    assert lib.lm_render_route(None, 4) < 0
    assert lib.lm_render_route(C.byref(_host_model(0, 1e-3)), 4) < 0
    assert lib.lm_render_route(C.byref(_host_model(64, 1e-3)), -1) < 0
