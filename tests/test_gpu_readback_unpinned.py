"""Arrays are read back where no pinned host memory is to be had (a process
whose hipHostMalloc, loaded before the library, refuses everything): the same
values as with it, from both solvers, small and large."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

RUN = """
import ctypes, hashlib, sys
if len(sys.argv) > 1:
    ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
from unsflow2d_amd import cc, meshgen, nc, nc_mesh
def show(name, a):
    print("array", name, a.shape, hashlib.sha256(a.tobytes()).hexdigest())
for nx, ny in ((12, 6), (400, 250)):
    s = cc.Solver(cc.Mesh.from_raw(meshgen.bump_channel(nx, ny, 7, h=0.05)), cc.Config(mach=0.55))
    s.keep_residual(True)
    s.iterate(2)
    for name in ("qc", "res", "dt", "la"):
        show(name, s.get(name))
    s = nc.NCSolver(nc.NCMesh.from_raw(nc_mesh.o_grid(nx, ny, 3, stretch=1.005 ** (999 / (ny - 1)))), timemode="rk3",
                    cfl_max=0.8)
    s.iterate(2)
    for name in ("qc", "dt"):
        show(name, s.get(name))
"""


def test_reads_without_pinned_memory(tmp_path):
    src, lib = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text("#include <stddef.h>\nint hipHostMalloc(void** p, size_t n, unsigned f)"
                   "{ return 2; }\n")  # hipErrorOutOfMemory
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    out = []
    for args in ([], [str(lib)]):
        print(f"case: read-back {'without' if args else 'with'} pinned memory", flush=True)
        r = subprocess.run([sys.executable, "-c", RUN, *args], cwd=ROOT, capture_output=True,
                           text=True, timeout=100, env={**os.environ, "PYTHONPATH": ROOT})
        assert r.returncode == 0, r.stderr
        out.append([ln for ln in r.stdout.splitlines() if ln.startswith("array")])
    assert len(out[0]) == 12
    assert out[0] == out[1]
