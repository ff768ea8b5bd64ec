"""The FP64 one-launch stage of inviscid M1 / M2 against the separate
face-flux and update launches of the per-stage entry points: bit for bit,
the state, the RK register and the step's CFL / deltaT, over both slot forms
(geometry table, and a face's own data where a mesh has too many distinct
records), both M1 forms (weights that are symmetric, and that are not),
cells of 3 to 6 faces, and cell counts around the 64-cell slot groups and the
256-cell blocks."""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi, cases, meshgen
from test_gpu_fused import CASES as SMALL

pytestmark = pytest.mark.gpu


def _box(nx, ny, nz, **kw):
    """A hex box at rest with a seeded perturbation."""
    mesh = meshgen.box_3d(nx, nx=nx, ny=ny, nz=nz)
    prm = cases.base_params(dim=3, solver=0)
    prm["dt"] = 0.3 / cases.sound_speed(prm)
    n = mesh.n_cells
    c = cases.Case("box", mesh, prm, np.full(n, prm["p_inf"]), np.full(n, prm["T_inf"]), np.zeros((n, 3)))
    return sc.with_params(sc.seeded_perturbation(c, amp=1e-2), **kw)


def _vortex(nx, ny, **kw):
    return sc.with_params(cases.isentropic_vortex(nx=nx, ny=ny, solver=kw.pop("solver", 0)), **kw)


CASES = dict(SMALL)
CASES.update({
    # 2D and 3D at the edges of the slot groups and blocks
    "vortex_7x9": lambda: _vortex(7, 9),
    "vortex_8x8": lambda: _vortex(8, 8),
    "vortex_13x5_M2": lambda: _vortex(13, 5, solver=1),
    "vortex_17x15_adjust": lambda: _vortex(17, 15, adjust_dt=1, max_co=0.3),
    "vortex_16x16": lambda: _vortex(16, 16),
    # weights off one half in the last bits: flux_m1
    "vortex_61x47": lambda: _vortex(61, 47),
    "box_2x2x2": lambda: _box(2, 2, 2),
    "box_4x4x4_adjust": lambda: _box(4, 4, 4, adjust_dt=1, max_co=0.3),
    "box_13x5x1": lambda: _box(13, 5, 1),
    "box_11x7x9": lambda: _box(11, 7, 9),
    # more distinct face records than the table holds: a face's own data
    "annulus_M1_own_data": lambda: sc.with_params(
        cases.cylinder_2d(n_theta=96, n_quad=10, n_tri=10, solver=0, minmod=0, noise=1e-3, Ls_diam=2.0), mu=0.0),
    "annulus_M2_own_data": lambda: sc.with_params(
        cases.cylinder_2d(n_theta=96, n_quad=10, n_tri=10, solver=1, minmod=0, noise=1e-3, Ls_diam=2.0), mu=0.0),
    "ogrid_M1_cyclic_own_data": lambda: sc.ogrid(12, 20, 5, solver=0, minmod=0, mu=0.0),
})


@pytest.mark.parametrize("name", sorted(CASES))
def test_fused_stage_equals_separate_launches(name):
    print(f"[fused64] {name}", flush=True)
    c = CASES[name]()
    assert c.params["mu"] == 0.0 and c.params["solver"] < 2
    fused, ref, many = (capi.GpuSolver.from_case(c) for _ in range(3))
    dt = c.params["dt"]
    adjust = bool(c.params.get("adjust_dt"))
    steps = 3
    for _ in range(steps):
        fused.run(1)
        ref.prepare_for_timestep()
        for rk in range(c.params["rk_order"]):
            ref.prepare_for_RKstep(rk)
            ref.set_boundary_conditions()
            ref.calc_gradients()
            ref.one_rk_step(rk, dt)
        if adjust:
            dt = ref.compute_dt(c.params["max_co"])
            assert fused.info().dt == dt
        assert np.array_equal(fused.q(), ref.q(), equal_nan=True)
        assert np.array_equal(fused.field(capi.FIELD_DQ), ref.field(capi.FIELD_DQ), equal_nan=True)
    if not adjust:
        assert fused.info().cfl == ref.compute_cfl(dt)
    # one call for all steps: the CFL reduction carried from step to step
    many.run(steps)
    assert np.array_equal(many.q(), fused.q(), equal_nan=True)
    assert many.info().cfl == fused.info().cfl and many.info().dt == fused.info().dt
    for g in (fused, ref, many):
        g.close()
