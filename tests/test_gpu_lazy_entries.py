"""A solver whose steps are one-launch stages holds no gather entries until a call
reads them: creation and runs leave them out of device_bytes, the first such call
adds them (16 B per 2D cell, 24 per 3D cell in whole groups of 64), gradients the
cells they lead to as well, and each of those calls gives what a solver gives that
never ran a one-launch stage."""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi

pytestmark = pytest.mark.gpu

CASES = {"vortex": lambda **kw: sc.vortex(19, solver=0, **kw),
         "box": lambda **kw: sc.seeded_perturbation(sc.box(7, solver=1, **kw))}


def _entries(c):
    n = c.n_cells
    return 16 * n if c.params["dim"] == 2 else 24 * ((n + 63) // 64 * 64)


@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_FP32P])
@pytest.mark.parametrize("name", sorted(CASES))
def test_entries_come_with_the_call_that_reads_them(name, prec):
    print(f"[lazy entries] {name} {prec}", flush=True)
    c = CASES[name]()
    s, ref = (capi.GpuSolver.from_case(c, precision=prec) for _ in range(2))

    def stages(v):
        v.prepare_for_timestep()
        for rk in range(c.params["rk_order"]):
            v.prepare_for_RKstep(rk)
            v.set_boundary_conditions()
            v.one_rk_step(rk, c.params["dt"])

    s.run(130)
    b0 = s.info().device_bytes
    s.run(100)  # nothing more, replays or not
    assert s.info().device_bytes == b0
    for _ in range(230):
        stages(ref)
    dt = c.params["dt"]
    assert s.compute_cfl(dt) == ref.compute_cfl(dt)
    assert s.compute_dt(0.3) == ref.compute_dt(0.3)
    assert s.info().device_bytes == b0 + (_entries(c) if prec == capi.PREC_FP32P else 0)
    stages(s)
    stages(ref)
    assert s.info().device_bytes == b0 + _entries(c)
    assert np.array_equal(s.q(), ref.q())
    for v in (s, ref):
        v.calc_VIS()
    assert s.info().device_bytes >= b0 + 2 * _entries(c)
    assert np.array_equal(s.field(capi.FIELD_DUDX), ref.field(capi.FIELD_DUDX))
    s.run(3)
    ref.run(3)
    assert np.array_equal(s.q(), ref.q())
    s.close()
    ref.close()


@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_FP32P])
def test_forces_and_groups_after_one_launch_stages(prec):
    """Wall forces and a group of one take the separate launches."""
    print(f"[lazy entries] forces, group {prec}", flush=True)
    c = sc.cylinder(24, solver=0, minmod=0, mu=0.0, have_res=0)
    s, ref = (capi.GpuSolver.from_case(c, precision=prec) for _ in range(2))
    ref.post_configure(have_forces=True)
    s.run(3)
    ref.run(3)
    s.post_configure(have_forces=True)
    s.run(4)
    ref.run(4)
    assert np.array_equal(s.q(), ref.q())
    s.close()
    a = capi.GpuSolver.from_case(c, precision=prec)
    a.run(7)
    g = capi.PartGroup([a])
    g.run(2)
    g.synchronize()
    ref.post_configure()
    ref.run(2)
    assert np.array_equal(a.q(), ref.q())
    g.close()
    a.close()
    ref.close()


def test_batch_of_solvers_that_ran_alone():
    print("[lazy entries] batch", flush=True)
    c = CASES["vortex"]()
    a, lone = (capi.GpuSolver.from_case(c, precision=capi.PREC_FP32P) for _ in range(2))
    a.run(5)
    b = capi.Batch()
    b.set([a])
    b.run(3)  # five stages: the first is separate launches
    b.synchronize()
    lone.run(8)
    assert np.array_equal(a.q(), lone.q())
    b.close()
    a.close()
    lone.close()
