"""The plan of the one-workgroup LU-SGS sweeps, replayed on the host (no GPU).

The sweep kernel has no check of its own: that every LDS slot it reads holds
the neighbour meant, that no slot is overwritten while another wave may still
read it, that a record fetched from memory is old enough to have arrived
there, and that the four waves meet at the same barriers, all follow from the
plan (csrc/sweep_plan.h).  native/sweep_plan_replay.cpp walks the plan step by
step and checks each of these, on levels of every width around a pass (64
nodes) and a step (256), on numberings that read far behind the ring, and on
nodes with any number of neighbours.
"""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "unsflow2d_amd", "csrc")


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    assert shutil.which("g++"), "g++ builds the replay"
    exe = str(tmp_path_factory.mktemp("replay") / "sweep_plan_replay")
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.environ.get("ROCM_PATH", "/opt/rocm") + "/include", "-I", CSRC, "-o",
                    exe, os.path.join(ROOT, "tests", "native", "sweep_plan_replay.cpp")],
                   check=True)

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True)
        print(r.stdout, r.stderr)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return run


def _ring(header, name):
    with open(os.path.join(CSRC, header)) as f:
        return int(re.search(rf"constexpr int {name} = (\d+);", f.read()).group(1))


RINGS = {"cc": ("cc_kernels.h", "CC_SW_RING"), "nc": ("nc_kernels.h", "SW_RING")}


@pytest.mark.parametrize("graph", [
    "cells 1 1", "cells 3 2", "cells 200 100", "cells 300 290",
    "grid 3 2", "grid 40 16", "grid 600 300", "shuffled 100 60 1", "shuffled 300 150 2",
    "layers 1 40 0", "layers 1 3000 1400", "layers 63 60 25", "layers 64 60 30",
    "layers 65 60 20", "layers 255 30 7", "layers 256 30 6", "layers 257 30 9",
    "layers 1400 8 2"])
@pytest.mark.parametrize("solver", list(RINGS))
def test_plan_holds_what_the_kernel_relies_on(replay, solver, graph):
    replay(_ring(*RINGS[solver]), *graph.split())


# one node joined to all of a chain: at the end of the forward sweep it reads
# n - 1 nodes, all but the ring's last 1 280 from stored records -- 63, 64, 65
# and many more than a pass fetches; in front, the backward sweep does
@pytest.mark.parametrize("n", [1281 + 63, 1281 + 64, 1281 + 65, 1281 + 66, 2000, 5000])
@pytest.mark.parametrize("where", ["first", "middle", "last"])
def test_nodes_of_any_number_of_neighbours(replay, n, where):
    out = replay(_ring(*RINGS["nc"]), "hub", n, {"first": 0, "middle": n // 2, "last": n - 1}[where])
    spilt = max(int(m) for m in re.findall(r"(\d+) from memory", out))
    if where != "middle":
        assert spilt == max(0, n - 1 - 1280 - 64)


def test_no_plan_past_the_kernel_limits(replay):
    """More positions than the kernel's 32-bit offsets reach (2^27), or more
    neighbours of a node than its 15-bit count holds: the caller sweeps by
    level launches instead."""
    replay(_ring(*RINGS["nc"]), "limits")
