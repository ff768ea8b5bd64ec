"""Long runs replay several steps at a time as a captured graph; it is captured
by a run that goes on past some 500 launches and rebuilt when what its launches
depend on changes.  States, CFL / deltaT, residuals and step counts equal the
same steps taken one run(1) call at a time, bit for bit, also with work between
the replays: a state set from outside, another deltaT, an odd number of single
steps (which swaps the state buffers), averages switched on and off."""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi

pytestmark = pytest.mark.gpu

CASES = {
    "vortex_M1": lambda: sc.vortex(16, solver=0),
    "vortex_M1_rk4": lambda: sc.vortex(16, solver=0, rk_order=4),
    "vortex_M2_res_adjust": lambda: sc.vortex(16, solver=1, rk_order=3, have_res=1, adjust_dt=1, max_co=0.2),
    "box_M1": lambda: sc.box(5, solver=0),
    "cylinder_M2AUSM_sponge_res": sc.PARITY_CASES["cylinder_M2AUSM_sponge"],
    "ogrid_M1_cyclic_rk2": sc.PARITY_CASES["ogrid_M1_cyclic_rk2"],
}


def _same(a, b, what):
    assert np.array_equal(a.q(), b.q(), equal_nan=True), what
    ia, ib = a.info(), b.info()
    assert (ia.cfl, ia.dt, ia.steps_done) == (ib.cfl, ib.dt, ib.steps_done), what


@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_FP32P])
@pytest.mark.parametrize("name", sorted(CASES))
def test_graph_replays_equal_single_steps(name, prec):
    print(f"[graph] {name} {prec}", flush=True)
    c = CASES[name]()
    many, one = (capi.GpuSolver.from_case(c, precision=prec) for _ in range(2))
    q0 = one.q()

    def both(n):
        many.run(n)
        for _ in range(n):
            one.run(1)

    both(240)  # past the capture, with replays
    _same(many, one, "first run")
    for n in (41, 3, 42, 19):  # replays with single steps before and after
        both(n)
        _same(many, one, n)
    if c.params["have_res"]:
        assert np.array_equal(many.residual(), one.residual())
    for g in (many, one):  # a state set from outside: its ghosts are filled first
        g.set_field(capi.FIELD_Q, q0)
    both(30)
    _same(many, one, "set state")
    if not c.params["adjust_dt"]:
        for g in (many, one):  # another deltaT, by the per-stage calls
            g.prepare_for_timestep()
            for rk in range(c.params["rk_order"]):
                g.prepare_for_RKstep(rk)
                g.set_boundary_conditions()
                g.calc_VIS()
                g.one_rk_step(rk, 0.5 * c.params["dt"])
        both(300)  # rebuilt on the way
        _same(many, one, "other deltaT")
    for g in (many, one):  # averages: no replays
        g.post_configure(have_average=True)
    both(12)
    assert np.array_equal(many.average_fields(12)[0], one.average_fields(12)[0], equal_nan=True)
    for g in (many, one):
        g.post_configure()
    both(25)
    _same(many, one, "after averages")
    many.close()
    one.close()


def test_batch_graphs_equal_lone_runs():
    print("[graph] batch", flush=True)
    mk = [lambda: sc.vortex(16, solver=2, minmod=1, mu=0.02), lambda: sc.vortex(20, solver=2, minmod=1, mu=0.02)]
    members = [capi.GpuSolver.from_case(f(), precision=capi.PREC_FP32P) for f in mk]
    b = capi.Batch()
    b.set(members)
    b.run(150)  # past the capture of several steps
    b.run(13)
    b.synchronize()
    lone = [capi.GpuSolver.from_case(f(), precision=capi.PREC_FP32P) for f in mk]
    for g, l in zip(members, lone):
        l.run(163)
        _same(g, l, "batch")
    b.set(members[:1])
    b.run(70)
    b.synchronize()
    lone[0].run(70)
    _same(members[0], lone[0], "one left")
    b.close()
    for g in members + lone:
        g.close()
