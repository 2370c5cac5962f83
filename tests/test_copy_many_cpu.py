"""CPU test of tsph_copy_many's refusals that need no device: a size that one
launch cannot cover (2^24 blocks of 16 KB, 256 GiB), among them those whose
number of blocks would wrap round to none."""
import ctypes

import pytest


@pytest.mark.parametrize("sizes", [[2 ** 64 - 1], [16, 2 ** 64 - 16383], [1 << 60], [1 << 38], [1 << 37, 1 << 37]])
def test_sizes_past_one_launch_are_refused(sizes):
    from tichi_sph_amd import _lib
    lib = _lib.load()
    moves = (_lib.TsphCopy * len(sizes))()
    here = (ctypes.c_uint8 * 16)()
    for q, s in enumerate(sizes):
        moves[q] = (ctypes.addressof(here), ctypes.addressof(here), s)
    assert lib.tsph_copy_many(moves, len(sizes), None) == -1
    assert b"too many bytes" in lib.tsph_last_error()
