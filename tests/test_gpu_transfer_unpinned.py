"""A handle on a system that pins no host memory: a child process whose
hipHostMalloc always fails (a library loaded before the engine's) makes
handles of every ring size and takes particles, accelerations and records
through ordinary memory, bit for bit."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = "int hipHostMalloc(void **p, unsigned long n, unsigned f) { *p = 0; calls++; return 2; }\n"

CHILD = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = [sys.argv[2], sys.argv[2] + "/tests"]
from cuco_amd import engine as E
from test_gpu_transfer import params
from test_gpu_transfer_rings import round_trip
for capacity, counts in ((341, (1, 341)), (21845, (20000,)), (300007, (5000, 131073, 300007)),
                         (1000001, (1000001,))):
    eng = E.Engine(max_particles=capacity, **params())
    for n in counts:
        print(capacity, n, flush=True)
        round_trip(eng, n, n)
    eng.close()
assert ctypes.c_int.in_dll(shim, "calls").value == 4
print("done", flush=True)
"""


def test_round_trips_without_pinned_memory(tmp_path):
    (tmp_path / "shim.c").write_text("int calls;\n" + SHIM)
    so = tmp_path / "shim.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(tmp_path / "shim.c"), "-o", str(so)],
                   check=True)
    out = subprocess.run([sys.executable, "-u", "-c", CHILD, str(so), ROOT], capture_output=True,
                         text=True, timeout=100, cwd=tmp_path, env=dict(os.environ))
    assert out.returncode == 0 and out.stdout.endswith("done\n"), out.stdout + out.stderr[-2000:]
