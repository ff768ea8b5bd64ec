"""Per-stage calls with a deltaT that changes from call to call, queued one
after another without a wait: each stage uses its own call's deltaT, as when the
stream is waited for after every call."""
import numpy as np
import pytest

from lfm_public_amd import capi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("adjust", [0, 1])
@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_FP32P])
def test_queued_stages_use_their_own_dt(prec, adjust):
    print(f"[stage dt] {prec} {adjust}", flush=True)
    # large enough that a stage is still running when the next call is made
    c = cases.cylinder_2d(n_theta=512, n_quad=128, n_tri=192, solver=2)
    c.params["adjust_dt"] = adjust
    out = []
    for wait in (True, False):
        s = capi.GpuSolver.from_case(c, precision=prec)
        s.synchronize()
        s.prepare_for_timestep()
        for rk in range(c.params["rk_order"]):
            s.prepare_for_RKstep(rk)
            s.set_boundary_conditions()
            s.calc_VIS()
            s.one_rk_step(rk, c.params["dt"] * (1.0 - 0.1 * rk))
            if wait:
                s.synchronize()
        out.append(s.q())
        assert s.info().dt == c.params["dt"] * (1.0 - 0.1 * (c.params["rk_order"] - 1))
        s.close()
    assert np.all(np.isfinite(out[0]))
    assert np.array_equal(out[0], out[1])
