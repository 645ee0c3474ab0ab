"""Whole RK3 iterations of the vertex-centred solver (one gradient and one
residual pass, three updates) against its stages one by one (a gradient and a
residual pass each, NCFVM/main.f90:51-88).

Primitives are refreshed once per iteration, so the stages' residuals are the
same numbers; every expression is evaluated uncontracted in both, so the
results are the same bits, in FP64 and in the mixed form.  Sizes: below one
block of 256 vertices, one block exactly, one over, several.  (AUSM+-up in the
mixed form turns non-finite on the 8 x 3 grid, stages and whole alike.)
"""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("ni,nj", [(8, 3), (16, 16), (57, 9), (40, 16)])
def test_whole_iterations_equal_the_stages(ni, nj, precision):
    from unsflow2d_amd import nc, nc_mesh
    m = nc.NCMesh.from_raw(nc_mesh.o_grid(ni, nj, 6, stretch=1.15))
    for grad, flux, limiter, order in (("gg", "vanleer", "vkn", "reference"),
                                       ("lsqr", "vanleer", "bj", "reference"),
                                       ("gg", "ausm", "bj", "multicolour"),
                                       ("lsqr", "ausm", "vkn", "reference")):
        print(f"case: nc whole rk3 vs stages, {ni}x{nj} {precision} {grad} {flux} {limiter}",
              flush=True)
        out = []
        for whole in (True, False):
            s = nc.NCSolver(m, mach=0.5, aoa_deg=1.5, cfl_max=0.8, grad=grad, timemode="rk3",
                            flux=flux, limiter=limiter, lusgs_order=order, precision=precision)
            if whole:
                hist = s.iterate(4)
            else:
                hist = []
                for it in range(1, 5):
                    # NCFVM/main.f90:54
                    cfl = 0.5 * 0.8 * (1.0 + math.tanh(it * 7.0 / 500.0 - 3.5))
                    s.save_old()
                    for k in (1, 2, 3):
                        s.rk_stage(k, cfl)
                    hist.append(s.residue(it))
            out.append([np.array(hist)] + [s.get(n) for n in ("qc", "qold", "res", "phi", "grad",
                                                               "qp", "la", "dt")])
        for a, b in zip(*out):
            assert np.array_equal(a, b, equal_nan=True)
