"""Whole laminar RK3 iterations with the diamond-path gradient (the interior
inviscid residual and the viscous fluxes per unit viscosity evaluated once)
against the stages one by one (CCFVM/main.F90:88-109, viscous_flux.F90).

Sizes: all cells at a boundary, one block of 256 cells, a few, and enough that
most blocks have no boundary cell; quadrilaterals; both wall conditions, with
and without the residual smoothing; every stage form.

Tolerance: the same expressions on the same numbers, up to the contraction of
products (a last bit per operation): 1e-12 normwise in FP64; one FP32 rounding
of a flux in the mixed form: 1e-6.
"""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu

MESHES = {"3x3": (3, 3, "tri"), "8x16": (8, 16, "tri"), "33x5": (33, 5, "tri"),
          "quad 16x17": (16, 17, "quad"), "90x80": (90, 80, "tri")}
CFL = 0.5


def routines(s, n):
    hist = []
    for it in range(1, n + 1):
        s.prim()
        s.avg_c2v()
        s.time_step(CFL)
        s.save_old()
        s.gradient()
        for k in (1, 2, 3):
            s.rk_stage(k)
        hist.append(s.residue(it)[0])
    return np.array(hist)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("irs,iwall", [(1, 1), (0, 0), (0, 1)])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_whole_iterations_equal_the_stages(mesh, irs, iwall, precision, tol):
    from unsflow2d_amd import cc, meshgen
    nx, ny, cells = MESHES[mesh]
    m = cc.Mesh.from_raw(meshgen.bump_channel(nx, ny, 7, h=0.05, cells=cells))
    for form in ("gather_lds", "shared") if mesh != "8x16" else ("gather", "gather_lds", "shared",
                                                                "shared_lds"):
        print(f"case: laminar whole vs stages, {mesh} {form} irs {irs} iwall {iwall} {precision}",
              flush=True)
        out = []
        for whole in (True, False):
            s = cc.Solver(m, cc.Config(mach=0.3, flow_type="laminar", reynolds=1000.0, iwall=iwall,
                                       grad="ggfc", irs=irs, cfl_min=CFL, cfl_max=CFL,
                                       precision=precision))
            s.set_stage_form(form)
            h = s.iterate(2) if whole else routines(s, 2)
            f = s.forces()
            out.append([h] + [s.get(n) for n in ("qc", "res", "phi", "fc_mu", "cell_mul", "qp")] +
                       [np.array([f["fx1"], f["fy1"]])])
        for a, b in zip(out[0][:-1], out[1][:-1]):
            assert np.all(np.isfinite(b))
            assert relerr(a, b) <= tol
        # the walls' pressure forces (p 7.9, length 3 each) mostly cancel
        assert np.abs(out[0][-1] - out[1][-1]).max() <= tol * 7.9 * 6
