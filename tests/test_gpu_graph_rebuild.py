"""A step graph that is rebuilt while replays of the one before may still be
queued: the calls follow one another without a wait, a step with another deltaT
between the runs, and the state equals the same steps taken one by one with a
wait after each."""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_FP32P])
def test_rebuilt_while_replays_are_queued(prec):
    print(f"[graph rebuild] {prec}", flush=True)
    c = sc.vortex(96, solver=0)
    queued, waited = (capi.GpuSolver.from_case(c, precision=prec) for _ in range(2))

    def other_dt(s, f):
        s.prepare_for_timestep()
        for rk in range(c.params["rk_order"]):
            s.prepare_for_RKstep(rk)
            s.set_boundary_conditions()
            s.one_rk_step(rk, f * c.params["dt"])

    for f in (0.5, 0.25, 0.125):
        queued.run(220)
        other_dt(queued, f)
    queued.run(20)
    for f in (0.5, 0.25, 0.125):
        for _ in range(220):
            waited.run(1)
            waited.synchronize()
        other_dt(waited, f)
    waited.run(20)
    assert queued.replayed_steps() > 0
    assert np.array_equal(queued.q(), waited.q())
    assert queued.info().dt == waited.info().dt
    queued.close()
    waited.close()
