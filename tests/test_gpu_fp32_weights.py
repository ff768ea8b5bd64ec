"""Face weights of the FP32 path keep their relative precision: between a cell of
width 1 and one of width 1e-5 the wide cell's weight is 1e-5, and with only the
wide cell off the freestream the face value is that product alone.  Velocity and
temperature gradients and the mass flux of the narrow cells against FP64, per
cell, to 1e-5: a dozen roundings of 2^-24 of either's value (weights held to
2^-25 absolutely would be off by 3e-3).  2D through the gather entries, 3D
through the slots; the M1 flux by the one-launch stage and by the separate
launches.  (A weight just below 1 has no such precision left in 1 - w: the narrow
cells compared are those whose wide neighbour is the face's P.)"""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi, cases, meshgen

pytestmark = pytest.mark.gpu

N = 12


def _case(dim, mu):
    """Columns of width 1 and 1e-5 in turn; every fourth (wide) column moves and
    is warmer."""
    mesh = meshgen.cartesian_2d(N, 3, 0, N, 0, 3, thickness=1.0) if dim == 2 else meshgen.box_3d(N, nx=N, ny=3, nz=3)
    edges = np.concatenate([[0.0], np.cumsum([1.0 if i % 2 == 0 else 1e-5 for i in range(N)])])
    x = mesh.points[:, 0]
    mesh.points[:, 0] = edges[np.rint(x - x.min()).astype(int)]
    prm = cases.base_params(dim=dim, solver=0, mu=mu, rk_order=1)
    prm["dt"] = 1e-6 / cases.sound_speed(prm)
    n = mesh.n_cells
    col = np.searchsorted(edges, meshgen.cell_centres_approx(mesh)[:, 0]) - 1
    wide = col % 4 == 0
    U = np.zeros((n, 3))
    U[wide, 0], U[wide, 1] = 0.1, 0.05
    T = np.where(wide, 1.01, 1.0) * prm["T_inf"]
    p = prm["p_inf"] * np.where(wide, 1.01, 1.0)  # the freestream's density
    return cases.Case("weights", mesh, prm, p, T, U), col % 4 == 1


def _close(a, b, what):
    assert np.all(b != 0) and np.all(np.abs(a - b) <= 1e-5 * np.abs(b)), (what, np.abs(a / b - 1).max())


@pytest.mark.parametrize("dim", [2, 3])
def test_gradients_of_narrow_cells(dim):
    print(f"[weights] gradients {dim}D", flush=True)
    c, narrow = _case(dim, 1e-3)
    v = []
    for prec in (capi.PREC_FP64, capi.PREC_FP32P):
        s = capi.GpuSolver.from_case(c, precision=prec)
        s.set_boundary_conditions()
        s.calc_VIS()
        v.append((s.field(capi.FIELD_DUDX), s.field(capi.FIELD_DTDX)))
        s.close()
    for k, i in ((0, 0), (0, dim), (1, 0)):  # du/dx, dv/dx, dT/dx
        _close(v[1][k][i][narrow], v[0][k][i][narrow], (k, i))


@pytest.mark.parametrize("dim", [2, 3])
def test_m1_flux_of_narrow_cells(dim):
    print(f"[weights] flux {dim}D", flush=True)
    c, narrow = _case(dim, 0.0)
    drho = []
    for prec, staged in ((capi.PREC_FP64, False), (capi.PREC_FP32P, False), (capi.PREC_FP32P, True)):
        s = capi.GpuSolver.from_case(c, precision=prec)
        if staged:
            s.prepare_for_timestep()
            s.prepare_for_RKstep(0)
            s.set_boundary_conditions()
            s.one_rk_step(0, c.params["dt"])
        else:
            s.run(1)
        drho.append(s.field(capi.FIELD_DQ)[0][narrow])
        s.close()
    _close(drho[1], drho[0], "one launch")
    assert np.array_equal(drho[1], drho[2])
