"""Which density calls sort their points first follows from the tables and the number of points; asked on the host, nothing is
launched.  The wrapper does not ask below 2^20 points."""
import ctypes as C
import os

import pytest

from landmark_amd import _lib as L


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(L.SO_PATH):
        from landmark_amd import build

        build.build(verbose=False)
    return L.load()


def _planes(n, channels, res=512, dtype=L.LM_F32):
    arr = (L.LmPlane * n)()
    for k in range(n):
        arr[k].plane = arr[k].line = 16
        arr[k].H = arr[k].W = arr[k].Len = res
        arr[k].C, arr[k].dtype = channels, dtype
        arr[k].ax0, arr[k].ax1, arr[k].axl = [(0, 1, 2), (0, 2, 1), (1, 2, 0)][k % 3]
    return arr


@pytest.mark.parametrize("n,channels,res,dtype,M,sorts", [
    (12, 64, 512, L.LM_F32, (1 << 20) - 1, False),  # the widest tables
    (12, 64, 512, L.LM_F32, 1562500, True), (12, 64, 512, L.LM_F32, 1562499, False),
    (3, 64, 2048, L.LM_F32, 6250000, True), (3, 64, 2048, L.LM_F32, 6249999, False), (3, 16, 1000, L.LM_F32, 25000000, True),
    (3, 64, 2048, L.LM_F16, 1 << 24, False), (3, 48, 2048, L.LM_F32, 1 << 24, False), (3, 64, 128, L.LM_F32, 1 << 24, False),
    (3, 16, 8192, L.LM_F32, 30000000, False)])  # fewer points than texels
def test_density_calls_that_sort(lib, n, channels, res, dtype, M, sorts):
    assert (lib.lm_gather_density_workspace_bytes(_planes(n, channels, res, dtype), n, M) > 0) == sorts
