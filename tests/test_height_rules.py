"""Rules that pick a tile height by the grid (functions of libphx.so, called by their C++ names; without a device they
count the 256 CUs of an MI355X)."""
import ctypes

import pytest


def dp45_rows(tetm, fp32, N_c, N_r):
    from phoenix_amd import _lib
    f = _lib.lib()._ZN3phx23dp45_adaptive_tile_rowsEbbii  # phx::dp45_adaptive_tile_rows(bool, bool, int, int)
    f.argtypes = [ctypes.c_bool, ctypes.c_bool, ctypes.c_int, ctypes.c_int]
    return f(tetm, fp32, N_c, N_r)


@pytest.mark.parametrize("N_c", [4096, 8192, 16384, 30000, 60000])
def test_dp45_height_reaches_no_further_than_32_rows(monkeypatch, N_c):
    """the largest FP32 TE-TM grids: what 32-row tiles take (their stores address, and drop, 32 + 7 rows past the
    grid's end) the chosen height takes too"""
    monkeypatch.delenv("PHX_GEN_TY", raising=False)
    limit = 2 ** 31 - 1
    last = limit // (8 * N_c) - 32 - 7  # rows of the largest such grid
    for N_r in range(last - 40, last + 1):
        ty = dp45_rows(True, True, N_c, N_r)
        assert N_c * (N_r + ty + 7) * 8 <= limit, (N_c, N_r, ty)


def test_dp45_heights_of_ordinary_grids(monkeypatch):
    monkeypatch.delenv("PHX_GEN_TY", raising=False)
    assert dp45_rows(True, True, 2048, 2048) == 42 and dp45_rows(True, True, 1024, 1024) == 28
    assert dp45_rows(True, True, 600, 600) == 8
