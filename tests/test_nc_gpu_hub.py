"""Reference-order LU-SGS on a mesh whose first and last vertices have 1 500
neighbours each, more than the sweep's LDS ring and one pass's fetch slots
hold: the sweep in one workgroup against the sweep by level launches (no ring,
no slots), bit for bit."""
import numpy as np
import pytest


def _two_hubs(n, seed):
    """Two vertices left and right of an upright curve of ``n`` vertices, each
    joined to all of them: the breadth-first numbering takes the left one
    first and the right one last.  The left edges of the outline are walls."""
    from unsflow2d_amd import nc_mesh
    rng = np.random.default_rng(seed)
    y = np.linspace(-1.0, 1.0, n)
    y[1:-1] += rng.uniform(-0.2, 0.2, n - 2) * (2.0 / n)
    x = 0.02 * (1.0 - y * y)
    xs = np.concatenate(([-1.0], x, [1.0]))
    ys = np.concatenate(([0.0], y, [0.0]))
    a = np.arange(1, n)
    left = np.stack([np.zeros_like(a), a, a + 1], 1)
    right = np.stack([np.full_like(a, n + 1), a + 1, a], 1)
    pbc = np.full(n + 2, nc_mesh.FARFIELD, dtype=np.int32)
    pbc[[0, 1, n]] = nc_mesh.WALL

    def ccw(t):
        d = ((xs[t[:, 1]] - xs[t[:, 0]]) * (ys[t[:, 2]] - ys[t[:, 0]]) -
             (xs[t[:, 2]] - xs[t[:, 0]]) * (ys[t[:, 1]] - ys[t[:, 0]]))
        return np.where((d < 0)[:, None], t[:, [0, 2, 1]], t)
    return nc_mesh._from_triangles(xs, ys, pbc, ccw(np.concatenate([left, right]).astype(np.int64)))


def _mesh(n):
    from unsflow2d_amd import nc
    m = nc.NCMesh.from_raw(_two_hubs(n, 11))
    cnt = m.get("pt_nv2v")
    assert cnt[0] == n and cnt[-1] == n  # both sweeps end with one
    return m


def test_hubs_are_numbered_first_and_last():
    _mesh(1500)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1300, 1345, 1346, 1500])
def test_one_workgroup_sweep_of_hubs_equals_the_levels(n, monkeypatch):
    from unsflow2d_amd import nc
    m = _mesh(n)
    qs = {}
    for mode in ("levels", "stream"):
        print(f"case: nc sweep with two hubs of {n} neighbours, {mode}", flush=True)
        monkeypatch.setenv("UFX_NC_SWEEP", mode)
        s = nc.NCSolver(m, mach=0.4, cfl_max=2.0, grad="gg", timemode="lusgs")
        s.iterate(3, hist=False)
        qs[mode] = s.get("qc")
        s.close()
    assert np.all(np.isfinite(qs["levels"]))
    np.testing.assert_array_equal(qs["stream"], qs["levels"])
