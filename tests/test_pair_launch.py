"""The FP32 pair force's launch sizes (tile_parts.h), compiled for the host:
the tuned workgroups per compute unit bound every launch, of a tile per wave
and of a tile per workgroup alike."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import ROOT

SOURCE = """
#include "tile_parts.h"
extern "C" uint32_t waves(uint32_t t, uint32_t w, uint32_t l) { return cuco::wave_tile_workgroups(t, w, l); }
extern "C" uint32_t team(uint32_t t, uint32_t l) { return cuco::team_tile_workgroups(t, l); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("launch")
    src, so = d / "launch.cpp", d / "launch.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "cuco_amd", "csrc"), str(src), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.waves.restype = lib.team.restype = C.c_uint32
    return lib


@pytest.mark.parametrize("per_cu", [1, 2, 8, 32])
@pytest.mark.parametrize("tiles", [0, 1, 255, 512, 513, 4096, 1 << 20])
@pytest.mark.parametrize("ncu", [32, 256])
def test_the_tuning_bounds_every_launch(lib, per_cu, tiles, ncu):
    limit = per_cu * ncu
    assert lib.team(tiles, limit) == max(1, min(tiles, 512, limit))
    assert lib.waves(tiles, 4, limit) == min(max(256, -(-tiles // 4)), limit)
