"""The transfer ring's host side on the CPU (ring_host.cpp): slots, events,
held chunks, errors on the way, rings handed from one handle to the next,
handles on several threads, and memory that the system will not pin."""
import os
import subprocess

import pytest

from conftest import ROOT

from cuco_amd import build


def test_ring_against_a_runtime_of_threads(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("needs hipcc to compile the host side")
    exe = tmp_path / "ring_host"
    cmd = [build.HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-I", build.INCLUDE,
           "-I", build.CSRC, os.path.join(ROOT, "tests", "ring_host.cpp"),
           os.path.join(build.CSRC, "transfer.hip"), "-c"]
    subprocess.run(cmd, check=True, cwd=tmp_path)
    # Only the runtime of the test is linked; the kernels' binary is never read.
    subprocess.run(["g++", "ring_host.o", "transfer.o", "-o", str(exe), "-lpthread",
                    "-no-pie", "-Wl,--unresolved-symbols=ignore-all"], check=True, cwd=tmp_path)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout[-2000:] + out.stderr[-500:]
