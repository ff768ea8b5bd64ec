"""The fixed-width gather entries (a cell's first four in 2D, six in 3D, with
placeholders past a shorter list and the rest from the gather list) at the
sizes where they can go wrong: cell counts below, at and past a wave of 64 and
a block of 256, 2D cells of 3 to 6 faces, 3D cells of 5, and cells that are
their own neighbour (eight entries).  FP64 against the oracle (relative L2 of
p, U and T <= 1e-10, as for every FP64 case), FP32 against FP64 (1e-5 of the
perturbation); the CFL and residual sums walk the same entries."""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi
from test_gpu_fp32p import _errors
from test_gpu_fp64 import _compare_prims, _pair

pytestmark = pytest.mark.gpu

CASES = {
    "poly_3x3": lambda: sc.poly(nx=3, ny=3, solver=2, mu=0.02, minmod=1, have_res=1),
    "poly_13x5": lambda: sc.poly(nx=13, ny=5, solver=2, mu=0.02, minmod=1, have_res=1),
    "poly_17x16": lambda: sc.poly(nx=17, ny=16, solver=1, mu=0.02, have_res=1),
    "vortex_8x8": lambda: sc.vortex(8, solver=2, mu=0.02, minmod=1, have_res=1),
    "vortex_16x16": lambda: sc.vortex(16, solver=0, mu=0.02, have_res=1),
    "cylinder_16": lambda: sc.cylinder(n_theta=16),
    "prism_3x3x3": lambda: sc.prism(nx=3, ny=3, nz=3, solver=2, mu=0.02, minmod=1, have_res=1),
    "prism_9x5x4": lambda: sc.prism(nx=9, ny=5, nz=4, solver=0, mu=0.02, have_res=1),
    "ogrid_own_neighbour": lambda: sc.ogrid(nr=6, nth=12, nz=1),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_gather_entries(name, oracle_lib):
    print(f"[keys] {name}", flush=True)
    case = CASES[name]()
    g, o = _pair(case, oracle_lib)
    g.run(4)
    o.run(4)
    assert np.all(np.isfinite(o.q()))
    for k, v in _compare_prims(case, g.q(), o.q()).items():
        assert v <= 1e-10, (k, v)
    assert g.info().cfl == pytest.approx(o.cfl, rel=1e-12)
    if case.params.get("have_res"):
        assert np.allclose(g.residual(), o.res(), rtol=1e-10, atol=0)
    if name != "ogrid_own_neighbour":  # FP32 takes at most six entries per cell
        f = capi.GpuSolver.from_case(case, precision=capi.PREC_FP32P)
        f.run(4)
        for k, v in _errors(case, f.q(), g.q()).items():
            assert v <= 1e-5, (k, v)
        assert f.info().cfl == pytest.approx(g.info().cfl, rel=1e-5)
        f.close()
    g.close()
