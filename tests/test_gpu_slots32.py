"""The FP32 face slots in both forms: packed words over the geometry table, and
a face's own data where a mesh has more distinct face records than the table
holds.  The one-launch stage against the separate launches of the per-stage
entry points, bit for bit, at cell counts around the 64-cell slot groups and
the 256-cell blocks; the 3D gradients, which read the same slots, against the
FP64 path to the FP32 path's 1e-5."""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi, cases
from test_gpu_fused64 import CASES as SHAPES

pytestmark = pytest.mark.gpu


def _annulus(solver):
    """4,864 cells, 7,744 jittered faces: more records than the table holds."""
    c = cases.cylinder_2d(n_theta=128, n_quad=10, n_tri=14, solver=solver, minmod=0, noise=1e-3, Ls_diam=2.0)
    return sc.with_params(c, mu=0.0)


CASES = {k: SHAPES[k] for k in ("vortex_7x9", "vortex_8x8", "vortex_13x5_M2", "vortex_17x15_adjust", "vortex_16x16",
                                "vortex_61x47", "box_2x2x2", "box_4x4x4_adjust", "box_13x5x1", "box_11x7x9")}
CASES.update({
    "annulus_M1_own_data": lambda: _annulus(0),
    "annulus_M2_own_data_adjust": lambda: sc.with_params(_annulus(1), adjust_dt=1, max_co=0.3),
    "ogrid_M1_cyclic_own_data": lambda: sc.ogrid(14, 24, 6, solver=0, minmod=0, mu=0.0),
})


@pytest.mark.parametrize("name", sorted(CASES))
def test_fused_stage_equals_separate_launches(name):
    print(f"[slots32] {name}", flush=True)
    c = CASES[name]()
    fused, ref = (capi.GpuSolver.from_case(c, precision=capi.PREC_FP32P) for _ in range(2))
    dt = c.params["dt"]
    adjust = bool(c.params.get("adjust_dt"))
    for _ in range(3):
        fused.run(1)
        ref.prepare_for_timestep()
        for rk in range(c.params["rk_order"]):
            ref.prepare_for_RKstep(rk)
            ref.set_boundary_conditions()
            ref.one_rk_step(rk, dt)
        if adjust:
            dt = ref.compute_dt(c.params["max_co"])
            assert fused.info().dt == dt
        assert np.array_equal(fused.q(), ref.q(), equal_nan=True)
        assert np.array_equal(fused.field(capi.FIELD_DQ), ref.field(capi.FIELD_DQ), equal_nan=True)
    if not adjust:
        assert fused.info().cfl == ref.compute_cfl(dt)
    fused.close()
    ref.close()


@pytest.mark.parametrize("name", ["box_packed", "ogrid_own_data"])
def test_3d_gradients_match_fp64(name):
    print(f"[slots32] gradients {name}", flush=True)
    c = (sc.seeded_perturbation(sc.box(7, solver=1, mu=1e-3)) if name == "box_packed"
         else sc.ogrid(14, 24, 6, solver=1, minmod=0))
    g = [capi.GpuSolver.from_case(c, precision=p) for p in (capi.PREC_FP64, capi.PREC_FP32P)]
    for v in g:
        v.run(2)
    for f in (capi.FIELD_DUDX, capi.FIELD_DTDX):
        a, b = (v.field(f) for v in g)
        assert np.linalg.norm(b - a) <= 1e-5 * np.linalg.norm(a)
    for v in g:
        v.close()
