"""Launch shapes of the persistent traversals (host arithmetic): a window of stack
rows that the caller chose takes no more LDS than its rows, so that more waves
reside; where a limit on the resident waves reserves LDS, stack rows fill it;
sizes are whole allocation granules, so that a grid computed from them resides."""
from __future__ import annotations

import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "aurora_amd", "csrc")
SRC = """
#include "launch_shape.h"
extern "C" uint32_t lds_for(uint32_t need, uint32_t blocks) { return (uint32_t)aur::lds_for_blocks(need, blocks); }
extern "C" void shape(uint32_t levels, uint32_t want, int chosen, uint32_t block, uint32_t waves, uint32_t* out) {
  const aur::StackShape s = aur::stack_shape(levels, want, chosen != 0, block, waves);
  out[0] = s.rows, out[1] = s.maxrows, out[2] = (uint32_t)s.lds;
}
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


@pytest.fixture(scope="module")
def shape(lib):
    def call(levels, want, chosen, block, waves):
        out = (ctypes.c_uint32 * 3)()
        lib.shape(levels, want, int(chosen), block, waves, out)
        return tuple(out)

    return call


def test_lds_is_whole_granules(lib):
    for blocks in range(1, 33):
        for need in (8, 512, 1280, 12288, 15360, 16384, 18432, 61440):
            lds = lib.lds_for(need, blocks)
            assert lds >= need and lds % GRANULE == 0
            assert lds < need + GRANULE or LDS // lds >= blocks


def test_every_row_of_17_levels(lib):
    """16 rows of 1 KB a block: 9 blocks reside, not 163840 / 16384."""
    assert LDS // lib.lds_for(16 * 1024, 10) == 9


def _granules(n):
    return (n + GRANULE - 1) // GRANULE * GRANULE


def _waves(lds, block):
    """Waves per CU that the LDS leaves room for."""
    assert lds == _granules(lds)  # else an occupancy computed from the size is too high
    return LDS // lds * block // 64


@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("waves", [16, 20, 24, 28])
def test_shapes(shape, block, waves):
    for levels in range(1, 31):
        need = max(levels - 1, 1)
        for want in (0, 1, 3, 10, 12, 15, 19, 29, 64):
            asked = need if want == 0 or want >= need else want
            # no limit: exactly the rows asked for
            assert shape(levels, want, True, block, 0) == (asked, need, _granules(asked * block * 8))
            rows, maxrows, lds = shape(levels, want, want != 0, block, waves)
            assert maxrows == need and rows * block * 8 <= lds
            if 0 < want < need:  # a chosen window keeps its rows and the residency they allow
                assert rows == want and lds == _granules(want * block * 8)
            else:
                assert rows == need and (lds == _granules(need * block * 8) or _waves(lds, block) >= waves - waves % (block // 64))
                # (a block of 64 is so small that the granules let a few more in)
                assert block == 64 or _waves(lds, block) <= waves
            # a default window fills the LDS that its residency reserves
            rows, _, lds = shape(levels, want, False, block, waves)
            assert asked <= rows <= need and rows * block * 8 <= lds and lds == _granules(lds)
            assert rows == need or lds - rows * block * 8 < block * 8


def test_batches_of_16_levels_need_no_split_stack(shape):
    assert shape(16, 12, False, 128, 20)[0] == 15


@pytest.mark.parametrize("rows,waves", [(12, 24), (10, 32), (15, 20)])
def test_residency_of_a_window(shape, rows, waves):
    assert _waves(shape(30, rows, True, 128, 20)[2], 128) == waves
