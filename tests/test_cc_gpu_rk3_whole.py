"""Whole inviscid RK3 iterations (one residual evaluation, three updates)
against the routines called one by one (a residual evaluation per stage).

The reference refreshes primitives, gradients and limiter values once per
iteration (CCFVM/main.F90:59-86), so the interior fluxes of its three stages
are the same numbers and only the wall faces follow the stage state
(CCFVM/boundCond.F90).  Sizes: around one and two blocks of 256 cells, around
64 boundary cells (one block of theirs), corner cells with two boundary faces,
quadrilaterals and mixed cells; every flux and kernel form.  Rusanov and
AUSM+-up run one iteration: with them the reference's scheme itself (and the
oracle) turns non-finite within three on these meshes, Rusanov through its
in-place conversion of the ghost state, AUSM+-up through its missing face
length.

Tolerance: both evaluate the same expressions; they may differ by the
contraction of products into fused operations, a last bit per operation, over
5 iterations: 1e-12 normwise in FP64; in the mixed form one FP32 rounding
(6e-8) of a flux: 1e-6.
"""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu

CFL = 0.8


def routines(s, n):
    hist = []
    for it in range(1, n + 1):
        s.prim()
        s.avg_c2v()
        s.time_step(CFL)
        s.save_old()
        s.gradient()
        for k in (1, 2, 3):
            s.fvresidual()
            s.rk_update(k)
        hist.append(s.residue(it)[0])
    return np.array(hist)


MESHES = {"8x16": (8, 16, "tri"), "9x14": (9, 14, "tri"), "16x16": (16, 16, "tri"),
          "33x5": (33, 5, "tri"), "3x3": (3, 3, "tri"), "quad 16x17": (16, 17, "quad"),
          "mixed 21x13": (21, 13, "mixed")}


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("form", ["gather", "gather_lds", "shared", "shared_lds"])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_whole_iterations_equal_the_routines(mesh, form, precision, tol):
    from unsflow2d_amd import cc, meshgen
    nx, ny, cells = MESHES[mesh]
    fluxes = {"roe": 5}
    if mesh in ("9x14", "mixed 21x13"):
        fluxes.update(vanleer=5, rusanov=1)
    if mesh == "9x14":
        fluxes.update(ausm=1)  # on the mixed cells the oracle is non-finite at once
    m = cc.Mesh.from_raw(meshgen.bump_channel(nx, ny, 7, h=0.05, cells=cells))
    for flux, n in fluxes.items():
        print(f"case: whole rk3 vs routines, {mesh} {form} {precision} {flux}", flush=True)
        out = []
        for whole in (True, False):
            s = cc.Solver(m, cc.Config(mach=0.55, aoa_deg=1.0, flux=flux, precision=precision))
            s.set_stage_form(form)
            s.keep_residual(True)
            h = s.iterate(n) if whole else routines(s, n)
            f = s.forces()
            out.append([h, s.get("qc"), s.get("res"), s.get("phi"),
                        np.array([f["cl1"], f["cd1"]])])
        for a, b in zip(*out):
            assert np.all(np.isfinite(b))
            assert relerr(a, b) <= tol


# A launch of both kinds of cells takes up to 512 blocks of 256 (FP64 gather
# form: those of the boundary cells, 64 to a block, counted in): 485, 527 and
# 514 blocks of cells and boundary cells, so that each form is on either side.
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("nx,ny", [(240, 250), (256, 255), (257, 256)])
def test_one_and_two_launches(nx, ny, precision, tol):
    from unsflow2d_amd import cc, meshgen
    m = cc.Mesh.from_raw(meshgen.bump_channel(nx, ny, 7, h=0.05))
    for form in ("gather_lds", "shared", "gather", "shared_lds"):
        print(f"case: whole rk3 vs routines, {nx}x{ny} {form} {precision}", flush=True)
        out = []
        for whole in (True, False):
            s = cc.Solver(m, cc.Config(mach=0.55, aoa_deg=1.0, precision=precision))
            s.set_stage_form(form)
            s.keep_residual(True)
            h = s.iterate(3) if whole else routines(s, 3)
            out.append([h, s.get("qc"), s.get("res"), s.get("phi")])
        for a, b in zip(*out):
            assert np.all(np.isfinite(b))
            assert relerr(a, b) <= tol
