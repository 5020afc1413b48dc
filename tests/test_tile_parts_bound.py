"""The list of tile parts (tile_parts.h) holds every part of any box, whatever
its work: the header, compiled for the host, against exact arithmetic.  A box's
work passes 2^32 shares from 1.4e14 candidates on."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

SOURCE = """
#include "tile_parts.h"
extern "C" uint32_t size(uint64_t total, uint32_t uniform) { return cuco::tile_part_size(total, uniform); }
extern "C" uint32_t parts(uint32_t e, uint32_t size) { return cuco::tile_parts(e, size); }
extern "C" uint64_t bound(uint64_t n, uint64_t nblocks) { return cuco::tile_parts_bound(n, nblocks); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("parts")
    src, so = d / "parts.cpp", d / "parts.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "cuco_amd", "csrc"), str(src), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.size.restype = lib.parts.restype = C.c_uint32
    lib.size.argtypes = [C.c_uint64, C.c_uint32]
    lib.parts.argtypes = [C.c_uint32, C.c_uint32]
    lib.bound.restype = C.c_uint64
    lib.bound.argtypes = [C.c_uint64, C.c_uint64]
    return lib


@pytest.mark.parametrize("total", [0, 4096, 1 << 27, (1 << 27) + 32767, 1 << 46, (1 << 47) - 1,
                                   1 << 47, (1 << 47) + (1 << 27), 10 ** 15, 10 ** 16, (1 << 64) - 1])
@pytest.mark.parametrize("uniform", [0, 5000, 10 ** 9])
def test_size_is_the_share_or_all_32_bits(lib, total, uniform):
    assert lib.size(total, uniform) == min(max(total // 32768, 4096, uniform), 2 ** 32 - 1)


@pytest.mark.parametrize("n,nblocks", [(64, 64), (300007, 1 << 15), (10 ** 8, 1 << 18),
                                       (2 ** 31 - 1, 1 << 24)])
@pytest.mark.parametrize("spread", ["all alike", "one block", "uneven"])
def test_every_part_has_its_place(lib, n, nblocks, spread):
    """Tiles of up to n estimated candidates each, from all in one block to
    evenly spread."""
    tiles = (n + 63) // 64
    if spread == "all alike":  # each meets all particles
        groups = [(tiles, n)]
    elif spread == "one block":
        groups = [(max(1, tiles // 2), n // 2), (tiles - tiles // 2, 100)]
    else:
        e = np.unique(np.geomspace(1, n, 40).astype(np.int64))
        groups = [(max(1, tiles // len(e)), int(x)) for x in e]
    total = sum(c * e for c, e in groups)
    size = lib.size(total, 0)
    listed = sum(c * lib.parts(e, size) for c, e in groups)
    assert listed <= lib.bound(n, nblocks)
