"""Rules that cut work into launches, checked on the host over all they accept."""
import ctypes

import pytest


@pytest.fixture(scope="module")
def lib():
    import chameleon_amd as ch
    return ch.load()


def test_norm_copy_pieces_divide_the_tile(lib):
    """The working copy walks a tile's column pieces eight columns at a time: a piece
    is a whole number of those, and the pieces are the tile.  The scratch of a call
    is (1 + pieces) NT^2 ldt doubles."""
    scratch = lib._ZN3chx1k23copy_lower_norm_scratchEii
    scratch.restype, scratch.argtypes = ctypes.c_size_t, [ctypes.c_int, ctypes.c_int]
    wrong = []
    for ldt in range(128, 2049, 128):
        for nt in range(1, 201):
            pieces, rest = divmod(scratch(nt, ldt), nt * nt * ldt)
            pieces -= 1
            if rest or pieces < 1 or ldt % pieces or (ldt // pieces) % 8:
                wrong.append((ldt, nt, pieces))
    assert not wrong, wrong[:10]
