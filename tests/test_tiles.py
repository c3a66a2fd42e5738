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


SIZES = ((16, 64), (32, 64), (64, 16), (64, 1024), (64, 4096), (128, 256), (256, 4), (256, 64), (256, 256), (4096, 1))


@pytest.fixture
def no_choice():
    """Leave every (kind, precision) without a choice afterwards."""
    yield
    for kind in KINDS:
        for precision in (M3P_FP64, M3P_MIXED):
            lib().m3p_set_stage2d_tile(kind, precision, *((64, 16) if kind == M3P_KIND_AMR_EULER2D else (256, 16)))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("precision", [M3P_FP64, M3P_MIXED])
def test_a_tile_choice_can_be_put_back(kind, precision, no_choice):
    """Read, set another shape, write back what was read: the library's own rule
    again, at every size; a pinned shape holds, whichever it is."""
    def rule():
        return [tile_of(kind, precision, n, nblk) for n, nblk in SIZES]

    def read():
        tj, h = ctypes.c_int(0), ctypes.c_int(0)
        assert lib().m3p_get_stage2d_tile(kind, precision, ctypes.byref(tj), ctypes.byref(h)) == 0
        return tj.value, h.value

    before, saved = rule(), read()
    for shape in ((64, 64), (32, 32), (16, 16), (64, 2)):
        assert lib().m3p_set_stage2d_tile(kind, precision, *shape) == 0
        assert read() == shape
        assert tile_of(kind, precision, 64, 1024) == (0,) + shape
        assert lib().m3p_set_stage2d_tile(kind, precision, *saved) == 0
        assert rule() == before and read() == saved
    # the shape that stands for no choice, as a choice
    assert lib().m3p_pin_stage2d_tile(kind, precision, *saved) == 0
    assert all(tile_of(kind, precision, 256, nblk) == (0,) + saved for nblk in (1, 16, 256))
    assert lib().m3p_set_stage2d_tile(kind, precision, *saved) == 0
    assert rule() == before
    assert lib().m3p_pin_stage2d_tile(kind, precision, 48, 16) == M3P_ERR_BAD_ARGUMENT


E, D, T = M3P_KIND_EULER2D, M3P_KIND_MINIDISK, M3P_KIND_AMR_EULER2D


@pytest.mark.parametrize("kind, precision, n, nblk, tile", [
    # strips of two, four and eight rows by the number of waves
    (E, M3P_FP64, 64, 127, (64, 2)), (E, M3P_FP64, 64, 128, (64, 4)), (E, M3P_FP64, 64, 255, (64, 4)),
    (E, M3P_FP64, 64, 256, (64, 8)), (E, M3P_MIXED, 64, 256, (64, 8)), (T, M3P_FP64, 64, 1408, (64, 8)),
    # sixteen rows in FP64 on meshes that fill the device
    (E, M3P_FP64, 64, 2047, (64, 8)), (E, M3P_FP64, 64, 2048, (64, 16)), (D, M3P_FP64, 256, 256, (64, 16)),
    (D, M3P_FP64, 4096, 1, (64, 16)), (T, M3P_FP64, 64, 4096, (64, 8)),
    # wide tiles in mixed precision
    (E, M3P_MIXED, 256, 127, (64, 8)), (E, M3P_MIXED, 256, 128, (256, 16)), (E, M3P_MIXED, 4096, 1, (256, 16)),
    (E, M3P_MIXED, 2048, 1, (64, 8)), (D, M3P_MIXED, 256, 63, (64, 8)), (D, M3P_MIXED, 256, 64, (256, 16)),
    (T, M3P_MIXED, 256, 256, (64, 8)), (E, M3P_FP64, 256, 64, (64, 8)),
    # blocks that only 128 divides, where 128 x 32 loads every CU alike
    (E, M3P_MIXED, 128, 255, (64, 8)), (E, M3P_MIXED, 128, 256, (128, 32)), (D, M3P_MIXED, 128, 256, (128, 32)),
    (D, M3P_MIXED, 128, 257, (64, 8)), (D, M3P_MIXED, 640, 16, (64, 8)), (D, M3P_MIXED, 128, 1024, (64, 8)),
    (T, M3P_MIXED, 128, 256, (64, 8)), (D, M3P_FP64, 128, 256, (64, 8)),
    # narrow blocks
    (E, M3P_FP64, 32, 64, (32, 4)), (E, M3P_FP64, 32, 4096, (32, 32)), (E, M3P_MIXED, 32, 4096, (32, 16)),
    (E, M3P_FP64, 16, 64, (16, 8)), (E, M3P_FP64, 48, 4096, (16, 16))])
def test_the_rule_by_size(kind, precision, n, nblk, tile):
    """The library's own choice on both sides of each line of the rule."""
    assert tile_of(kind, precision, n, nblk) == (0,) + tile
