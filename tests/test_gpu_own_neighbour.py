"""Cells that are their own neighbour (a cyclic pair one cell apart) on the FP32
path: such a face stands twice in the cell's gather list, so a 3D cell has eight
entries and a 2D cell six.  All of them count in fluxes, gradients and residual,
and each face once in the CFL, whatever order the patches have (cyclic patches
first puts other faces past the sixth entry).  FP32 against FP64 to the FP32
path's 1e-5 of the perturbation; FP64 against the oracle."""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi, cases, meshgen
from test_gpu_fp32p import _errors
from test_gpu_fp64 import _compare_prims, _pair

pytestmark = pytest.mark.gpu


def _ogrid(**kw):
    """One cell in the span, cyclic patches first, flow along the span."""
    c = sc.ogrid(nr=6, nth=12, nz=1, **kw)
    c.mesh = sc.reorder_patches(c.mesh, ["back", "front", "cylinder", "inlet", "outlet"])
    c.U[:, 2] += 0.5 * cases.sound_speed(c.params)
    return c


def _strip(**kw):
    """One column of cells between a cyclic pair, cyclic patches first."""
    mesh = meshgen.cartesian_2d(1, 40, 0.0, 1.0, 0.0, 40.0,
                                names=(("left", "cyclic"), ("right", "cyclic"), ("inlet", "patch"),
                                       ("outlet", "patch")))
    by = {p.name: p for p in mesh.patches}
    by["left"].neighbour, by["right"].neighbour = "right", "left"
    prm = cases.base_params(dim=2, solver=0)
    c_inf = cases.sound_speed(prm)
    prm["U_inf"] = (0.5 * c_inf, 0.3 * c_inf, 0.0)
    prm["mach"] = 0.58
    prm["dt"] = 0.2 / c_inf
    n = mesh.n_cells
    U = np.tile(np.array(prm["U_inf"]), (n, 1))
    c = cases.Case("strip", mesh, prm, np.full(n, prm["p_inf"]), np.full(n, prm["T_inf"]), U)
    return sc.with_params(sc.seeded_perturbation(c, amp=1e-2), **kw)


CASES = {
    "ogrid_M2AUSM": lambda: _ogrid(have_res=1),
    "ogrid_M1_visc": lambda: _ogrid(solver=0, minmod=0),
    "ogrid_M1_euler": lambda: _ogrid(solver=0, minmod=0, mu=0.0),
    "ogrid_M2_adjust": lambda: _ogrid(solver=1, minmod=0, mu=0.0, adjust_dt=1, max_co=0.3),
    "strip_M2AUSM": lambda: _strip(solver=2, minmod=1, mu=0.02, have_res=1),
    "strip_M1_euler": lambda: _strip(),
    "strip_M2_adjust": lambda: _strip(solver=1, adjust_dt=1, max_co=0.3),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_fp32_counts_every_entry(name, oracle_lib):
    print(f"[own neighbour] {name}", flush=True)
    c = CASES[name]()
    g, o = _pair(c, oracle_lib)
    f = capi.GpuSolver.from_case(c, precision=capi.PREC_FP32P)
    for s in (g, o, f):
        s.run(4)
    assert np.all(np.isfinite(g.q()))
    for k, v in _compare_prims(c, g.q(), o.q()).items():
        assert v <= 1e-10, (k, v)
    for k, v in _errors(c, f.q(), g.q()).items():
        assert v <= 1e-5, (k, v)
    assert f.info().dt == pytest.approx(g.info().dt, rel=1e-5)
    dt = g.info().dt
    assert f.compute_cfl(dt) == pytest.approx(g.compute_cfl(dt), rel=1e-5)
    assert f.compute_dt(0.3) == pytest.approx(g.compute_dt(0.3), rel=1e-5)
    if c.params.get("have_res"):
        assert np.allclose(f.residual(), g.residual(), rtol=1e-3)
    f.close()
    g.close()


def test_batch_of_such_members_equals_lone_runs():
    print("[own neighbour] batch", flush=True)
    mk = [lambda: _ogrid(solver=0, minmod=0, mu=0.0), lambda: _ogrid(solver=0, minmod=0, mu=0.0, rk_order=5)]
    members = [capi.GpuSolver.from_case(m(), precision=capi.PREC_FP32P) for m in mk]
    b = capi.Batch()
    b.set(members)
    b.run(5)
    b.synchronize()
    b.close()
    for m, s in zip(mk, members):
        lone = capi.GpuSolver.from_case(m(), precision=capi.PREC_FP32P)
        lone.run(5)
        assert np.array_equal(lone.q(), s.q())
        lone.close()
        s.close()
