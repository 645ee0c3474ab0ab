"""The reference-order LU-SGS sweeps in one workgroup against the same sweeps
level by level, one launch each (CCFVM/lusgs.F90:207-379).

A context made for LU-SGS sweeps in one workgroup; one made for RK3 whose
caller runs the lusgs routine launches the levels.  Sizes: fewer nodes than
one group of passes, levels just under and over the 64 nodes of a pass and
the 256 of a step, quadrilaterals and mixed cells (four swept neighbours),
and grids whose cells read neighbours that have left the LDS ring.

Tolerance: the sums of fluxes are formed in a different order, a few last
bits of a flux per cell, in updates that are a fraction of the state, over 4
iterations of a diagonally dominant sweep: 1e-12 normwise for the state; the
history's norms are differences of fluxes, about three digits below them:
1e-9.  The mixed form holds the state, the residual it sweeps and the sweeps
themselves in FP64, but an update that differs in its last bit can turn one
FP32 rounding (6e-8) of the next residual: 1e-6 and 1e-4.
"""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu

MESHES = {"1x1": (1, 1, "tri"), "3x2": (3, 2, "tri"), "40x20": (40, 20, "tri"),
          "63x64": (63, 64, "tri"), "200x100": (200, 100, "tri"), "quad 5x3": (5, 3, "quad"),
          "quad 65x64": (65, 64, "quad"), "quad 300x290": (300, 290, "quad"),
          "mixed 61x33": (61, 33, "mixed")}


@pytest.mark.parametrize("precision,tol,htol", [("fp64", 1e-12, 1e-9), ("mixed", 1e-6, 1e-4)])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_one_workgroup_equals_the_levels(mesh, precision, tol, htol):
    from unsflow2d_amd import cc, meshgen
    nx, ny, cells = MESHES[mesh]
    m = cc.Mesh.from_raw(meshgen.bump_channel(nx, ny, 7, h=0.05, cells=cells))
    out = []
    for timemode in ("lusgs", "rk3"):
        print(f"case: reference-order sweep, {mesh} {precision} {timemode}", flush=True)
        s = cc.Solver(m, cc.Config(mach=0.55, aoa_deg=1.0, timemode=timemode, cfl_min=5.0,
                                   cfl_max=5.0, precision=precision))
        hist = []
        for it in range(1, 5):
            s.prim()
            s.avg_c2v()
            s.time_step(5.0)
            s.save_old()
            s.gradient()
            s.lusgs()
            hist.append(s.residue(it)[0])
        out.append((s.get("qc"), np.array(hist)))
    (q, h), (rq, rh) = out
    assert np.all(np.isfinite(rq)) and np.all(np.isfinite(rh))
    assert relerr(q, rq) <= tol
    assert relerr(h, rh) <= htol
