"""The kernel variants that are chosen past the Infinity Cache (non-temporal marks,
six faces in flight in the FP64 3D gradients, records stored in groups of 16
cells, unpacked slots in the FP32 3D gradients), which small cases never reach: on
meshes just past the line, FP64 against the oracle (relative L2 of p, U and T <=
1e-10, as for every FP64 case), FP32 against FP64 (1e-5 of the perturbation, the
FP32 path's bar), one step each."""
import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi, cases
from test_gpu_fp32p import _errors
from test_gpu_fp64 import _compare_prims, _pair

pytestmark = pytest.mark.gpu


def _ogrid(nz, **kw):
    return cases.cylinder_3d(nr=96, nth=96, nz=nz, pert=0.05, **kw)


def _past_the_line(s, grad_values, word):
    """The stage's bytes, each array once (tests/test_stage_footprint.py)."""
    i = s.info()
    D = i.dim
    cell = (2 * (D + 2) + 2) * word + 2 * 4 * (4 if D == 2 else 6) + grad_values * word
    return i.n_cells * cell + i.n_faces * ((3 * D + 3) * word + 8) > 330e6


# values of a gradient record: dudx, dTdx, with M2AUSM rho and p (FP64 also U)
RECORD = {(64, 2): 14, (64, 3): 28, (32, 2): 10, (32, 3): 18}


def _record(c, prec):
    D = c.params["dim"]
    return RECORD[prec, D] if c.params["solver"] == 2 else D * D + D


FP64 = {
    "ogrid_M2AUSM": lambda: _ogrid(56, solver=2, minmod=1),
    "ogrid_M2AUSM_nominmod": lambda: _ogrid(56, solver=2, minmod=0),
    "ogrid_M1": lambda: _ogrid(66, solver=0, minmod=0),
    # cells of 4 to 6 faces
    "poly_M2AUSM": lambda: sc.poly(nx=900, ny=640, solver=2, mu=0.02, minmod=1),
}
FP32 = {
    "ogrid_M2AUSM": lambda: _ogrid(112, solver=2, minmod=1),
    "ogrid_M1": lambda: _ogrid(129, solver=0, minmod=0),
    # packed slots
    "box_M2_visc": lambda: cases.acoustic_box(n=106, solver=1, mu=1e-3, amp=1e-2),
    "poly_M2AUSM": lambda: sc.poly(nx=1200, ny=900, solver=2, mu=0.02, minmod=1),
}


@pytest.mark.parametrize("name", sorted(FP64))
def test_fp64_past_the_cache_matches_oracle(name, oracle_lib):
    c = FP64[name]()
    print(f"[marked] FP64 {name} {c.n_cells} cells", flush=True)
    g, o = _pair(c, oracle_lib)
    assert _past_the_line(g, _record(c, 64), 8)
    g.run(1)
    o.run(1)
    assert np.all(np.isfinite(o.q()))
    for k, v in _compare_prims(c, g.q(), o.q()).items():
        assert v <= 1e-10, (k, v)
    assert g.info().cfl == pytest.approx(o.cfl, rel=1e-12)
    g.close()


@pytest.mark.parametrize("name", sorted(FP32))
def test_fp32_past_the_cache_matches_fp64(name):
    c = FP32[name]()
    print(f"[marked] FP32 {name} {c.n_cells} cells", flush=True)
    g, f = (capi.GpuSolver.from_case(c, precision=p) for p in (capi.PREC_FP64, capi.PREC_FP32P))
    assert _past_the_line(f, _record(c, 32), 4)
    for s in (g, f):
        s.run(1)
    for k, v in _errors(c, f.q(), g.q()).items():
        assert v <= 1e-5, (k, v)
    assert f.info().cfl == pytest.approx(g.info().cfl, rel=1e-5)
    g.close()
    f.close()
