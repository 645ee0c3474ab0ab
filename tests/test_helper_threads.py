"""The read-back's helper threads (csrc/helper_threads.h) when one cannot be
started for lack of memory: the read goes on with those there are instead of
ending the process (no GPU)."""
import os
import subprocess

from conftest import ROOT


def test_threads_that_find_no_memory(tmp_path):
    exe = str(tmp_path / "helper_threads")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread",
                    "-I", os.path.join(ROOT, "unsflow2d_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "native", "helper_threads.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
