"""The pair force's table index (common.h), compiled for the host: every
distance of a pair, and the NaN that a distance of zero gives, converts to an
index inside the table and its one entry past the end."""
import ctypes as C
import math
import os
import subprocess

import pytest

from cuco_amd import build

SOURCE = """
#include "common.h"
extern "C" int index(double x) { return cuco::table_index64(x); }
"""


def test_index_is_in_range(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("needs hipcc to compile the host side")
    (tmp_path / "index.cpp").write_text(SOURCE)
    subprocess.run([build.HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-fPIC", "-I",
                    build.CSRC, "-c", "index.cpp"], check=True, cwd=tmp_path)
    subprocess.run(["g++", "-shared", "index.o", "-o", "index.so"], check=True, cwd=tmp_path)
    index = C.CDLL(str(tmp_path / "index.so")).index
    index.argtypes = [C.c_double]
    for x, want in [(0.0, 0), (5e-324, 0), (0.999, 0), (1.0, 1), (999.999, 999), (1000.0, 1000),
                    (1000.001, 1000), (2.0 ** 31, 1000), (1e300, 1000), (math.inf, 1000),
                    (math.nan, 1000), (-math.nan, 1000)]:
        assert index(x) == want, x
