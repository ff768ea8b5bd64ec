"""A step that another one follows in the same call leaves its RK register
unstored (the next step starts from zero); the call's last step stores it.
The register, the state and the CFL after run(n), a batch's run(n) and a
partition group's run(n) equal those of single-step calls, bit for bit, in
every kind of stage: one-launch and separate, 2D and 3D, one to five stages,
table and own face data, more faces than slots."""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi, cases, meshgen

pytestmark = pytest.mark.gpu

CASES = {
    "vortex_M1": lambda: sc.vortex(17, solver=0),
    "vortex_M2_rk1": lambda: sc.vortex(16, solver=1, rk_order=1),
    "vortex_M1_rk2_adjust": lambda: sc.vortex(16, solver=0, rk_order=2, adjust_dt=1, max_co=0.3),
    "poly_M1": lambda: sc.poly(solver=0),
    "box_M1": lambda: sc.seeded_perturbation(sc.box(7, solver=0)),
    "prism_M2_adjust": lambda: sc.prism(solver=1, adjust_dt=1, max_co=0.3),
    "poly_M2AUSM_visc_rk1": lambda: sc.poly(solver=2, mu=0.02, minmod=1, rk_order=1),
    "cylinder_M2AUSM_sponge": sc.PARITY_CASES["cylinder_M2AUSM_sponge"],
    "ogrid_M2AUSM_cyclic": sc.PARITY_CASES["ogrid_M2AUSM_cyclic"],
}


@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_FP32P])
@pytest.mark.parametrize("name", sorted(CASES))
def test_register_after_runs(name, prec):
    print(f"[rk register] {name} {prec}", flush=True)
    c = CASES[name]()
    many, one = (capi.GpuSolver.from_case(c, precision=prec) for _ in range(2))
    for n in (1, 2, 5):
        many.run(n)
        for _ in range(n):
            one.run(1)
        assert np.array_equal(many.q(), one.q(), equal_nan=True), n
        assert np.array_equal(many.field(capi.FIELD_DQ), one.field(capi.FIELD_DQ), equal_nan=True), n
        a, b = many.info(), one.info()
        assert (a.cfl, a.dt) == (b.cfl, b.dt), n
    many.close()
    one.close()


@pytest.mark.parametrize("solver", [0, 2])
def test_register_after_batch_runs(solver):
    print(f"[rk register] batch {solver}", flush=True)
    mk = [lambda: sc.vortex(16, solver=solver, minmod=1, mu=0.01 * solver),
          lambda: sc.vortex(20, solver=solver, minmod=1, mu=0.01 * solver)]
    members = [capi.GpuSolver.from_case(f(), precision=capi.PREC_FP32P) for f in mk]
    b = capi.Batch()
    b.set(members)
    b.run(128)  # single-step launches, then eight at a time
    b.run(16)
    b.synchronize()
    b.close()
    for m, f in zip(members, mk):
        lone = capi.GpuSolver.from_case(f(), precision=capi.PREC_FP32P)
        lone.run(144)
        assert np.array_equal(m.q(), lone.q())
        assert np.array_equal(m.field(capi.FIELD_DQ), lone.field(capi.FIELD_DQ))
        lone.close()
        m.close()


def test_register_after_group_runs():
    print("[rk register] group", flush=True)
    base = sc.with_params(sc.PARITY_CASES["cylinder_M2AUSM_sponge"](), have_res=0)
    runs = []
    for steps in ((4,), (1, 1, 1, 1)):
        pcs = cases.partition(base, meshgen.slab_ranks(base.mesh, 2, axis=0))
        gp = [capi.GpuSolver.from_case(pc) for pc in pcs]
        capi.connect(gp)
        grp = capi.PartGroup(gp)
        for n in steps:
            grp.run(n)
        grp.synchronize()
        runs.append([g.q() for g in gp] + [g.field(capi.FIELD_DQ) for g in gp])
        grp.close()
        for g in gp:
            g.close()
    for x, y in zip(*runs):
        assert np.array_equal(x, y)
