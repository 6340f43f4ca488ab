"""Launch shapes of the persistent traversals (host arithmetic): LDS sizes are whole
allocation granules, so that a grid computed from them resides."""
from __future__ import annotations

import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "aurora_amd", "csrc")
SRC = """
#include "launch_shape.h"
extern "C" uint32_t lds_for(uint32_t need, uint32_t blocks) { return (uint32_t)aur::lds_for_blocks(need, blocks); }
"""
LDS, GRANULE = 160 << 10, 1280


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("shape")
    (d / "shape.cpp").write_text(SRC)
    out = str(d / "shape.so")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}", "-o", out,
                    str(d / "shape.cpp")], check=True)
    return ctypes.CDLL(out)


def test_lds_is_whole_granules(lib):
    for blocks in range(1, 33):
        for need in (8, 512, 1280, 12288, 15360, 16384, 18432, 61440):
            lds = lib.lds_for(need, blocks)
            assert lds >= need and lds % GRANULE == 0
            assert lds < need + GRANULE or LDS // lds >= blocks


def test_every_row_of_17_levels(lib):
    """16 rows of 1 KB a block: 9 blocks reside, not 163840 / 16384."""
    assert LDS // lib.lds_for(16 * 1024, 10) == 9
