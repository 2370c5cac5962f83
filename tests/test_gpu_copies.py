"""GPU test of tsph_copy_many: several copies in one launch, of sizes around
its 16 KB chunks, at aligned, 4-byte and odd offsets, exact to the byte and
nothing beyond; and its refusals."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

CHUNK = 16384


@pytest.mark.parametrize("off", [0, 4, 1])
def test_copies_are_exact(off):
    from tichi_sph_amd import _lib
    lib = _lib.load()
    sizes = [0, 1, 15, 16, 17, 300, CHUNK - 1, CHUNK, CHUNK + 1, 3 * CHUNK + 20, 1 << 20]
    g = torch.Generator().manual_seed(off)
    src = [torch.randint(0, 256, (s + 64,), dtype=torch.uint8, generator=g).cuda() for s in sizes]
    dst = [torch.full((s + 64,), 7, dtype=torch.uint8, device="cuda") for s in sizes]
    moves = (_lib.TsphCopy * len(sizes))()
    for q, s in enumerate(sizes):
        moves[q] = (dst[q].data_ptr() + off, src[q].data_ptr() + (off if q % 2 else 0), s)
    stream = torch.cuda.current_stream().cuda_stream
    print(f"[case] {len(sizes)} copies at offset {off}", flush=True)
    assert lib.tsph_copy_many(moves, len(sizes), stream) == 0
    for q, s in enumerate(sizes):
        o = off if q % 2 else 0
        want = torch.full((s + 64,), 7, dtype=torch.uint8, device="cuda")
        want[off:off + s] = src[q][o:o + s]
        assert torch.equal(dst[q], want), s


def test_refusals():
    from tichi_sph_amd import _lib
    lib = _lib.load()
    moves = (_lib.TsphCopy * (_lib.COPY_MAX + 1))()
    assert lib.tsph_copy_many(moves, 0, None) == 0
    assert lib.tsph_copy_many(moves, _lib.COPY_MAX, None) == 0  # nothing to move
    assert lib.tsph_copy_many(moves, _lib.COPY_MAX + 1, None) == -1
    assert lib.tsph_copy_many(None, 1, None) == -1
    moves[0] = (None, None, 4)
    assert lib.tsph_copy_many(moves, 1, None) == -1
    assert ctypes.sizeof(_lib.TsphCopy) == 24
