"""A batch's graph of several steps takes every stage of an inviscid step as one
launch, also where a step has an odd number of stages (a single step's graph
then takes its first stage as separate launches): after runs that mix both, the
members equal lone runs bit for bit, for odd and even stage counts, 2D and 3D,
members of very different size and an unset patch whose ghosts are carried
between the two state buffers."""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi
from test_gpu_fused import _unset_patch

pytestmark = pytest.mark.gpu

CASES = {
    "vortex_rk5": [lambda: sc.vortex(9, solver=0), lambda: sc.vortex(40, solver=0), lambda: sc.vortex(16, solver=0)],
    "vortex_rk4": [lambda: sc.vortex(16, solver=1, rk_order=4), lambda: sc.vortex(24, solver=1, rk_order=4)],
    "vortex_rk1": [lambda: sc.vortex(16, solver=0, rk_order=1), lambda: sc.vortex(20, solver=0, rk_order=1)],
    "box_rk3": [lambda: sc.box(5, solver=0, rk_order=3), lambda: sc.box(7, solver=0, rk_order=3)],
    "cylinder_unset": [lambda: _unset_patch(sc.cylinder(n_theta=16, solver=1, minmod=0, mu=0.0, have_res=0)),
                       lambda: sc.cylinder(n_theta=32, solver=1, minmod=0, mu=0.0, have_res=0)],
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_graphs_of_several_steps_equal_lone_runs(name):
    print(f"[batch graph] {name}", flush=True)
    members = [capi.GpuSolver.from_case(f(), precision=capi.PREC_FP32P) for f in CASES[name]]
    b = capi.Batch()
    b.set(members)
    n = 0
    for k in (130, 17, 8, 3, 24):
        b.run(k)
        b.synchronize()
        n += k
    b.close()
    for f, m in zip(CASES[name], members):
        lone = capi.GpuSolver.from_case(f(), precision=capi.PREC_FP32P)
        for _ in range(n):
            lone.run(1)
        assert np.array_equal(lone.q(), m.q(), equal_nan=True)
        assert np.array_equal(lone.field(capi.FIELD_DQ), m.field(capi.FIELD_DQ), equal_nan=True)
        a, c = lone.info(), m.info()
        assert (a.cfl, a.steps_done) == (c.cfl, c.steps_done)
        lone.close()
        m.close()
