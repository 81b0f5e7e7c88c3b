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


# resident dposv in ms, tiles rounded up to 16 and to 64 (differences above 5 %)
PADDING = [(2000, 16, 29.49, 6.97), (2000, 17, 28.69, 6.53), (2000, 40, 12.30, 1.63), (4000, 16, 60.74, 38.65),
           (4000, 17, 62.59, 32.99), (4000, 32, 30.65, 6.90), (4000, 33, 32.13, 6.98), (4000, 40, 24.65, 4.48),
           (4000, 72, 14.99, 4.15), (4000, 80, 13.17, 3.42), (4000, 100, 11.40, 2.43), (4000, 200, 7.71, 2.22),
           (5500, 16, 83.73, 94.48), (5500, 17, 90.88, 79.18), (5500, 32, 41.64, 14.56), (8000, 16, 128.74, 275.04),
           (8000, 17, 164.81, 231.09), (8000, 32, 64.53, 38.73), (8000, 33, 78.72, 35.71), (8000, 40, 60.89, 21.30),
           (8000, 72, 36.86, 20.27), (8000, 80, 31.32, 15.13), (8000, 100, 29.00, 9.01), (11000, 16, 211.35, 701.52),
           (11000, 17, 301.50, 584.37), (11000, 32, 104.43, 94.99), (11000, 33, 133.65, 86.36),
           (11000, 40, 95.66, 50.18), (11000, 72, 59.12, 47.11), (11000, 80, 49.68, 35.56), (11000, 144, 36.08, 20.71),
           (16000, 32, 183.51, 274.87), (16000, 40, 190.40, 144.16), (16000, 72, 119.57, 133.60),
           (16000, 100, 99.44, 53.29), (16000, 200, 68.65, 49.62), (23000, 32, 375.51, 793.30),
           (23000, 72, 265.46, 374.87), (23000, 80, 208.25, 276.91), (23000, 100, 228.74, 146.14),
           (23000, 200, 162.14, 138.15), (23000, 272, 143.60, 109.24), (23000, 336, 142.62, 100.74)]


def test_padding_goes_where_it_was_faster(lib):
    rule = lib._ZN3chx13mirror_pads64Eii
    rule.restype, rule.argtypes = ctypes.c_bool, [ctypes.c_int, ctypes.c_int]
    wrong = [c for c in PADDING if rule(-(-c[0] // c[1]), -(-c[1] // 16) * 16) != (c[3] < c[2])]
    assert not wrong, wrong


def test_padding_is_bounded(lib):
    """Whole 64x64 blocks are left alone, and no mirror above 16 GiB is made for the rest."""
    rule = lib._ZN3chx13mirror_pads64Eii
    rule.restype, rule.argtypes = ctypes.c_bool, [ctypes.c_int, ctypes.c_int]
    for t in range(16, 2049, 16):
        for nt in (1, 2, 7, 30, 100, 400, 1500, 4000):
            if rule(nt, t):
                assert t % 64 and (nt * (-(-t // 64) * 64)) ** 2 * 8 <= 16 << 30


SWITCHES = ["CHAMELEON_TILE_SIZE", "CHAMELEON_INNER_BLOCK_SIZE", "CHAMELEON_TRANSLATION_MODE", "CHAMELEON_GERED_ACC",
            "CHAMELEON_LOOKAHEAD", "CHAMAMD_PAIRS", "CHAMAMD_PANEL", "CHAMAMD_SMALL_COLS", "CHAMAMD_PAD64",
            "CHAMAMD_FWD_TAIL", "CHAMAMD_SERVE_SMALL", "CHAMAMD_SERVE_LANES", "CHAMAMD_BATCH_GRAPHS",
            "CHAMAMD_XFER_THREADS", "CHAMAMD_XFER_ZC", "CHAMAMD_ATOMIC_UPDATE"]


@pytest.mark.parametrize("name", SWITCHES)
def test_documented_switches_are_read(name):
    """Every environment variable that the documents offer is named in a source."""
    import os
    import chameleon_amd as ch
    src = os.path.join(os.path.dirname(ch.LIB_PATH), "csrc")
    for folder, _, files in os.walk(src):
        for f in files:
            with open(os.path.join(folder, f)) as h:
                text = h.read()
            if '("%s"' % name in text:
                return
    raise AssertionError(name)
