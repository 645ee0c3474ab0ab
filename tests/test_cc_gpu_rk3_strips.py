"""Whole RK3 iterations on strips in which nearly every cell has a boundary
face, against the routines one by one.

The boundary cells are taken 64 at a time; where one launch takes both kinds of
cells a block goes through all those among its 256, here up to four rounds
(one of less than 64 cells, of exactly 64 and a few more among them), and the
LDS, the residual norm and the limiter's range carry over from round to round.

Tolerance: as the whole iterations on other meshes, the same expressions up to
the contraction of products, a last bit per operation over 5 iterations: 1e-12
normwise in FP64, one FP32 rounding of a flux in the mixed form: 1e-6.
"""
import numpy as np
import pytest

from conftest import relerr
from test_cc_gpu_rk3_whole import routines

pytestmark = pytest.mark.gpu

STRIPS = {"32x1": (32, 1, "tri"), "33x1": (33, 1, "tri"), "100x1": (100, 1, "tri"),
          "128x1": (128, 1, "tri"), "129x2": (129, 2, "tri"), "300x1": (300, 1, "tri"),
          "quad 150x2": (150, 2, "quad")}


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("form", ["gather", "gather_lds", "shared", "shared_lds"])
@pytest.mark.parametrize("strip", list(STRIPS))
def test_strips(strip, form, precision, tol):
    from unsflow2d_amd import cc, meshgen
    nx, ny, cells = STRIPS[strip]
    m = cc.Mesh.from_raw(meshgen.bump_channel(nx, ny, 7, h=0.05, cells=cells))
    print(f"case: whole rk3 vs routines, strip {strip} {form} {precision}", flush=True)
    out = []
    for whole in (True, False):
        s = cc.Solver(m, cc.Config(mach=0.55, aoa_deg=1.0, precision=precision))
        s.set_stage_form(form)
        s.keep_residual(True)
        h = s.iterate(5) if whole else routines(s, 5)
        out.append([h, s.get("qc"), s.get("res"), s.get("phi")])
    for a, b in zip(*out):
        assert np.all(np.isfinite(b))
        assert relerr(a, b) <= tol
