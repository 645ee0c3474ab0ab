"""Read-back of per-cell and per-vertex arrays (ufx_cc_get, ufx_nc_get): what
was injected comes back exactly, in the reference's numbering.

Injection permutes on the host, read-back on the device: up to 4 MB (131 072
rows of four doubles) in one copy, above that chunk by chunk with threads.
The sizes lie on both sides of that, on whole chunks and not, and above the
ring of pinned memory (16 MB).  Values are distinct, so a row in the wrong
place shows.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _values(shape, seed):
    n = int(np.prod(shape))
    return (np.random.default_rng(seed).permutation(n) + 0.25).reshape(shape)


@pytest.mark.parametrize("nx,ny", [(1, 1), (16, 15), (63, 64), (129, 131), (256, 256),
                                   (255, 258), (760, 380)])
def test_cell_arrays_come_back_as_injected(nx, ny):
    from unsflow2d_amd import cc, meshgen
    m = cc.Mesh.from_raw(meshgen.bump_channel(nx, ny, 7, h=0.05))
    for precision in ("fp64", "mixed"):
        print(f"case: cc read-back {nx}x{ny} {precision}", flush=True)
        s = cc.Solver(m, cc.Config(mach=0.5, precision=precision))
        for name in ("la", "qc", "qold", "res", "dt", "qc"):  # grows and shrinks
            a = _values(s.get(name).shape, len(name))
            s.set(name, a)
            assert np.array_equal(s.get(name), a), name


@pytest.mark.parametrize("ni,nj", [(8, 3), (64, 64), (301, 157), (520, 260), (1000, 550)])
def test_vertex_arrays_come_back_as_injected(ni, nj):
    from unsflow2d_amd import nc, nc_mesh
    print(f"case: nc read-back {ni}x{nj}", flush=True)
    m = nc.NCMesh.from_raw(nc_mesh.o_grid(ni, nj, 3, stretch=1.005 ** (999.0 / (nj - 1))))
    s = nc.NCSolver(m, mach=0.4, timemode="rk3", cfl_max=0.8)
    for name in ("qc", "qold"):
        a = _values(s.get(name).shape, len(name))
        s.set(name, a)
        assert np.array_equal(s.get(name), a), name
