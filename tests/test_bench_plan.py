"""The benchmark's launch plan against the committed profiles: every kernel it
names, up to the parameters that depend on the mesh, is one kernel of its
workload's traffic summary, so that the measured bytes are found."""
import json
import os

import pytest

import bench
from lfm_public_amd import cases

PROFILES = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles")

WORKLOADS = {
    "vortex256x256": lambda: cases.isentropic_vortex(nx=4),
    "cylinder2d_1048576": lambda: cases.cylinder_2d(n_theta=8, n_quad=2, n_tri=3, solver=2),
    "cyl3d_256x256x64": lambda: cases.cylinder_3d(nr=4, nth=8, nz=2, solver=1, minmod=1),
    "box256": lambda: cases.acoustic_box(n=3),
}


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("key", sorted(WORKLOADS))
def test_every_planned_kernel_is_in_the_profile(key, precision):
    prm = dict(WORKLOADS[key]().params, precision=precision)
    with open(os.path.join(PROFILES, f"{key}_traffic.json")) as f:
        names = list(json.load(f)["kernels"])
    plan = bench.launch_plan(prm, prm["rk_order"])
    assert plan
    for group, (n, kernel) in plan.items():
        if n:
            assert len([k for k in names if k.startswith(kernel)]) == 1, (group, kernel)
            assert bench.traffic_of(key, kernel)[0] > 0, (group, kernel)
