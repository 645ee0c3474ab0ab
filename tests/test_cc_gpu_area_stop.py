"""The diamond-path area stop (CCFVM/gradient.F90:297) inside a whole
iteration: the primitives are refreshed before the gradient that fails, as in
the reference (CCFVM/main.F90:62-86), and are read back as the iteration
started from them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("flow,irs", [("inviscid", 0), ("laminar", 1)])
def test_primitives_after_an_area_stop(flow, irs, precision):
    from unsflow2d_amd import cc, meshgen
    print(f"case: area stop, {flow} {precision}", flush=True)
    good = cc.Mesh.from_raw(meshgen.bump_channel(40, 20, 7, h=0.05))
    a = good.arrays()
    f = 700  # an interior face seen from its other side: both its triangles turn over
    for k in ("fc_p1", "fc_p2"):
        a[k] = a[k].copy()
    a["fc_p1"][f], a["fc_p2"][f] = a["fc_p2"][f], a["fc_p1"][f]
    m = cc.Mesh.import_arrays(a, len(a["fc_p1"]) - (len(a["cell_cenx"]) - len(a["cell_cv"])))
    out = []
    for mesh, grad in ((m, "ggfc"), (good, "lsqr")):
        s = cc.Solver(mesh, cc.Config(mach=0.5, flow_type=flow, irs=irs, grad=grad,
                                      precision=precision))
        q = s.get("qc")
        noc = s.counts["noc"]
        q[:noc] *= 1.0 + 0.01 * np.random.default_rng(5).uniform(-1.0, 1.0, (noc, 4))
        s.set("qc", q)
        if grad == "ggfc":
            with pytest.raises(cc.UfxError, match="-ve area"):
                s.iterate(1)
            assert s.error()["kind"] == "area" and s.error()["face"] == f + 1
        else:
            s.prim()
        out.append(s.get("qp")[:noc])
    np.testing.assert_array_equal(*out)
