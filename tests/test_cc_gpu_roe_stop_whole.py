"""Roe stops of whole RK3 iterations.

The reference loops over the boundary faces before the interior ones
(CCFVM/fvresidual.F90:27-190) and stops at the first whose Roe average has no
speed of sound (CCFVM/roe_flux.F90:73-87).  A whole iteration evaluates both
kinds at once or the interior ones first, so a failure met in one must not keep
the others from being evaluated: the face reported is the oracle's, and the
state of every cell away from the failures is that of an iteration without
them, whatever the order in which the device came to the cells.

Cells of negative pressure are planted in a channel's disturbed stream; the same
form of the kernels runs with and without them, so away from them (without the
limiter, whose range is global) the bits are the same.  The meshes are below
and above the 512 blocks of one launch for both kinds of cells; both precisions,
the four forms, a batch and a captured chunk.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MACH = 0.5


def _mesh(nx, ny):
    from unsflow2d_amd import cc, meshgen
    return cc.Mesh.from_raw(meshgen.bump_channel(nx, ny, 7, h=0.05))


def _cells(arrs, nx, ny):
    """A cell at the wall and one in the interior, well apart, and the
    distance of all cells from the nearer of them in cell widths."""
    noc = len(arrs["cell_cv"])
    x, y = arrs["cell_cenx"][:noc], arrs["cell_ceny"][:noc]
    nof, nbf = len(arrs["fc_p1"]), len(arrs["cell_cenx"]) - noc
    bc = np.asarray(arrs["fc_bc"])[nof - nbf:]
    inner = np.asarray(arrs["fc_in"])[nof - nbf:] - 1
    walls = inner[bc == 1001] if np.any(bc == 1001) else inner[bc == 1]
    xm = x.min() + 0.25 * (x.max() - x.min())
    wall = int(walls[np.argmin(np.abs(x[walls] - xm))])
    xi = x.min() + 0.75 * (x.max() - x.min())
    inside = int(np.argmin((x - xi) ** 2 + (y - 0.5 * (y.min() + y.max())) ** 2))
    w = np.sqrt(np.max(arrs["cell_cv"]))
    dist = np.minimum(np.hypot(x - x[wall], y - y[wall]), np.hypot(x - x[inside], y - y[inside]))
    return wall, inside, dist / w


def _disturbed(q):
    return q * (1.0 + 0.01 * np.random.default_rng(5).uniform(-1.0, 1.0, q.shape))


def _plant(q, cells):
    q = q.copy()
    for c in cells:
        q[c, 0] = -5.0 * abs(q[c, 0])
    return q


def _solver(m, form, precision, ilimit):
    from unsflow2d_amd import cc
    s = cc.Solver(m, cc.Config(mach=MACH, precision=precision, ilimit=ilimit))
    s.set_stage_form(form)
    return s


def _oracle_face(arrs, q, ilimit):
    from oracle.oracle import CCOracle
    orc = CCOracle(arrs, mach=MACH, ilimit=ilimit)
    orc.qc[:] = q
    with pytest.raises(RuntimeError):
        orc.iteration(1, 0.8)
    assert orc.error_info["kind"] == 1
    return orc.error_info["face"], orc.error_info["cell"]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("form", ["gather", "gather_lds", "shared", "shared_lds"])
@pytest.mark.parametrize("nx,ny", [(40, 20), (257, 256)])
def test_boundary_and_interior_failures(nx, ny, form, precision):
    from unsflow2d_amd.cc import UfxError
    m = _mesh(nx, ny)
    arrs = m.arrays()
    wall, inside, dist = _cells(arrs, nx, ny)
    nbf = len(arrs["cell_cenx"]) - len(arrs["cell_cv"])
    nfi = len(arrs["fc_p1"]) - nbf
    for ilimit in (1, 0):
        for cells in ((wall, inside), (inside,)):
            print(f"case: Roe stop, {nx}x{ny} {form} {precision} ilimit {ilimit} cells {cells}",
                  flush=True)
            s = _solver(m, form, precision, ilimit)
            q0 = _disturbed(s.get("qc"))
            q = _plant(q0, cells)
            face, cell = _oracle_face(arrs, q, ilimit)
            assert (face > nfi) == (len(cells) == 2)
            s.set("qc", q)
            with pytest.raises(UfxError):
                s.iterate(1)
            want = dict(kind="roe", face=face, cell=cell)
            assert s.error() == want
            got = s.get("qc")[:len(dist)]
            # later iterations do no work
            with pytest.raises(UfxError):
                s.iterate(3)
            assert s.error() == want
            np.testing.assert_array_equal(s.get("qc")[:len(dist)], got)
            s.close()
            if ilimit == 0:
                h = _solver(m, form, precision, ilimit)
                h.set("qc", q0)
                h.iterate(1)
                away = dist > 8.0
                assert away.sum() > 0.5 * len(dist)
                np.testing.assert_array_equal(got[away], h.get("qc")[:len(dist)][away])
                h.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_and_captured_chunk(precision):
    from unsflow2d_amd import cc
    from unsflow2d_amd.cc import UfxError
    m = _mesh(40, 20)
    arrs = m.arrays()
    wall, inside, _ = _cells(arrs, 40, 20)
    print(f"case: Roe stop in a batch and a captured chunk, {precision}", flush=True)
    ss = [_solver(m, "gather_lds", precision, 1) for _ in range(3)]
    for k in ss:
        k.iterate(1)
    q = _plant(_disturbed(ss[1].get("qc")), (wall, inside))
    face, cell = _oracle_face(arrs, q, 1)
    want = dict(kind="roe", face=face, cell=cell)
    ss[1].set("qc", q)
    b = cc.Batch(ss)
    with pytest.raises(UfxError, match="case 1"):
        b.iterate(4)
    assert ss[1].error() == want
    assert ss[0].error()["kind"] is None and ss[2].error()["kind"] is None
    s = _solver(m, "gather_lds", precision, 1)
    s.iterate(1)
    s.set("qc", q)
    with pytest.raises(UfxError):
        s.iterate_graph(4)
    assert s.error() == want
