"""bench.py names the kernel behind every stage time: small chunks have fused kernels, whose time falls into one interval."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

from landmark_amd import _lib as L


@pytest.mark.parametrize("route,kernels", [(0, ["k_march", "k_app_feat", "k_mlp"]), (L.LM_ROUTE_RAYS, ["k_rays", "k_app_feat", "k_mlp"]),
                                           (L.LM_ROUTE_RAYS | L.LM_ROUTE_SHADE, ["k_rays", "k_shade"])])
def test_stage_intervals_belong_to_the_kernels_that_ran(route, kernels):
    import bench

    got = bench.stage_kernels(route)
    assert [k for _, _, k in got] == kernels
    covered = [i for _, at, _ in got for i in at]
    assert len(covered) == len(set(covered)) and set(covered) >= {1, 3, 4}  # no interval twice, no gather or network left out
    assert all(nm in L.STAGE_NAMES and nm == L.STAGE_NAMES[at[0]] for nm, at, _ in got)
