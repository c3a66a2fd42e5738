"""The 2D stage tiles: which shape a stage takes, and the block sizes it
refuses (host state and host arithmetic: no device needed)."""
import ctypes

import pytest

from mara3p_amd._lib import (M3P_ERR_BAD_ARGUMENT, M3P_ERR_BAD_SHAPE, M3P_FP64, M3P_KIND_AMR_EULER2D,
                             M3P_KIND_EULER2D, M3P_KIND_MINIDISK, M3P_MIXED, lib)

KINDS = (M3P_KIND_EULER2D, M3P_KIND_MINIDISK, M3P_KIND_AMR_EULER2D)


def tile_of(kind, precision, n, nblk):
    """(status, columns, rows) of a stage over nblk blocks of n x n zones."""
    tj, h = ctypes.c_int(0), ctypes.c_int(0)
    st = lib().m3p_stage2d_tile(kind, precision, n, nblk, ctypes.byref(tj), ctypes.byref(h))
    return st, tj.value, h.value


@pytest.mark.parametrize("n", [0, -16, -32, -64, -256, 1, 8, 24, 72])
def test_unusable_block_sizes_have_no_tile(n):
    """Zero and negative sizes are refused like any other that no tile divides."""
    for kind in KINDS:
        for precision in (M3P_FP64, M3P_MIXED):
            assert tile_of(kind, precision, n, 4)[0] == M3P_ERR_BAD_SHAPE
    assert tile_of(M3P_KIND_EULER2D, M3P_FP64, 64, 0)[0] == M3P_ERR_BAD_ARGUMENT


@pytest.mark.parametrize("n", [16, 32, 48, 64, 80, 96, 128, 192, 256, 320, 512, 1024, 4096])
@pytest.mark.parametrize("nblk", [1, 16, 1024, 65536])
def test_every_block_size_has_a_tile_that_divides_it(n, nblk):
    for kind in KINDS:
        for precision in (M3P_FP64, M3P_MIXED):
            st, tj, h = tile_of(kind, precision, n, nblk)
            assert st == 0 and n % tj == 0 and n % h == 0, (kind, precision, tj, h)
