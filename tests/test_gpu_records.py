"""The gradient pass stores whole records (primitives, limiter values,
gradient, centroid) through LDS, 32 or 64 rows at a time: node counts around
multiples of 32, 64 and 256, against the oracle.

Tolerances: those of the routine-by-routine tests (cell-centred: the kernels
contract products into fused operations, 1e-12 normwise; vertex-centred: the
same bits).
"""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,cells", [(31, 1, "quad"), (16, 2, "quad"), (11, 3, "quad"),
                                         (21, 3, "quad"), (16, 4, "tri"), (13, 5, "quad"),
                                         (51, 5, "quad"), (16, 8, "tri"), (43, 3, "tri")])
@pytest.mark.parametrize("grad", ["lsqr", "gg", "ggfc"])
def test_cell_records(nx, ny, cells, grad):
    from unsflow2d_amd import cc, meshgen
    from oracle.oracle import CCOracle
    print(f"case: cc records {nx}x{ny} {cells} {grad}", flush=True)
    m = cc.Mesh.from_raw(meshgen.bump_channel(nx, ny, 5, h=0.05, cells=cells))
    dev = cc.Solver(m, cc.Config(mach=0.5, grad=grad))
    orc = CCOracle(m.arrays(), mach=0.5, grad=grad)
    q = orc.qc * (1.0 + 0.01 * np.random.default_rng(1).uniform(-1, 1, orc.qc.shape))
    dev.set("qc", q)
    orc.qc[:] = q
    for s in (dev, orc):
        s.prim()
        s.avg_c2v()
        s.time_step(0.8)
        s.save_old()
        s.gradient()
        s.fvresidual()
    for n in ("grad", "phi", "res"):
        assert relerr(dev.get(n), getattr(orc, n)) <= 1e-12, n


@pytest.mark.parametrize("ni,nj", [(11, 3), (16, 2), (21, 3), (16, 4), (13, 5), (85, 3), (64, 4),
                                   (43, 6)])
@pytest.mark.parametrize("grad", ["gg", "lsqr"])
def test_vertex_records(ni, nj, grad):
    from unsflow2d_amd import nc, nc_mesh
    from oracle.oracle import NCOracle
    print(f"case: nc records {ni}x{nj} {grad}", flush=True)
    m = nc.NCMesh.from_raw(nc_mesh.o_grid(ni, nj, 3, stretch=1.1))
    dev = nc.NCSolver(m, mach=0.4, cfl_max=0.8, grad=grad, timemode="rk3")
    orc = NCOracle(m.arrays(), mach=0.4, cfl_max=0.8, grad=grad)
    q = orc.qc * (1.0 + 0.01 * np.random.default_rng(1).uniform(-1, 1, orc.qc.shape))
    dev.set("qc", q)
    orc.qc[:] = q
    dev.save_old(); orc.save_old()
    dev.fvresidual(0.3); orc.fvresidual(0.3)
    for n in ("qp", "phi", "grad", "res"):
        assert np.array_equal(dev.get(n), getattr(orc, n)), n


@pytest.mark.parametrize("nx,ny,cells", [(3, 3, "tri"), (16, 17, "quad"), (129, 131, "tri"),
                                         (256, 256, "tri"), (257, 256, "tri")])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_face_radii(nx, ny, cells, precision):
    """The face radii that the gradient pass forms on meshes of up to 512
    blocks of 256 cells (131 072), against the routine's own pass: nothing in
    them is contracted, so they, the cells' radii and the time steps are the
    same bits."""
    from unsflow2d_amd import cc, meshgen
    m = cc.Mesh.from_raw(meshgen.bump_channel(nx, ny, 5, h=0.05, cells=cells))
    for grad in ("lsqr", "gg"):
        print(f"case: face radii {nx}x{ny} {cells} {grad} {precision}", flush=True)
        cfg = cc.Config(mach=0.5, grad=grad, precision=precision, cfl_min=0.8, cfl_max=0.8)
        whole, parts = cc.Solver(m, cfg), cc.Solver(m, cfg)
        q = whole.get("qc")
        q[:, :] *= 1.0 + 0.01 * np.random.default_rng(1).uniform(-1, 1, q.shape)
        for s in (whole, parts):
            s.set("qc", q)
        whole.iterate(1)
        parts.prim()
        parts.avg_c2v()
        parts.time_step(0.8)
        for n in ("fc_la", "la", "dt"):
            assert np.array_equal(whole.get(n), parts.get(n)), n
