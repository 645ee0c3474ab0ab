"""Vertex averages (CCFVM/average.F90:11-29) against the oracle where a vertex
has up to, exactly and more than the eight cells whose list entries are loaded
slot by slot: a fan of n triangles around one vertex.

Tolerance: the device contracts products into fused operations (a last bit an
operation over at most 40 terms): 1e-13 normwise.
"""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu


def fan(n):
    from unsflow2d_amd import meshgen
    a = 2.0 * np.pi * np.arange(n) / n
    r = 1.0 + 0.1 * np.random.default_rng(n).uniform(size=n)
    xs = np.r_[0.0, r * np.cos(a)]
    ys = np.r_[0.0, r * np.sin(a)]
    k = np.arange(n)
    tri = np.stack([np.zeros(n, np.int64), 1 + k, 1 + (k + 1) % n], 1)
    return meshgen._from_triangles(xs, ys, np.zeros(n + 1, np.int32), tri,
                                   wall_of=lambda p, q: (ys[p] < 0) & (ys[q] < 0))


@pytest.mark.parametrize("n", [5, 8, 9, 12, 40])
def test_averages_of_a_fan(n):
    from unsflow2d_amd import cc
    from oracle.oracle import CCOracle
    print(f"case: vertex averages, fan of {n}", flush=True)
    m = cc.Mesh.from_raw(fan(n))
    orc = CCOracle(m.arrays(), mach=0.5)
    q = orc.qc * (1.0 + 0.01 * np.random.default_rng(1).uniform(-1, 1, orc.qc.shape))
    orc.qc[:] = q
    orc.prim()
    orc.avg_c2v()
    for precision, tol in (("fp64", 1e-13), ("mixed", 1e-6)):
        dev = cc.Solver(m, cc.Config(mach=0.5, precision=precision))
        dev.set("qc", q)
        dev.prim()
        dev.avg_c2v()
        assert relerr(dev.get("pt_prim"), orc.pprim) <= tol
