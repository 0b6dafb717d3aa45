"""Products of 32-bit matrices refuse strides and depths whose offsets in a tile
do not fit 32 bits, before anything of the GPU is asked for."""
import ctypes

import pytest
import torch

import llmlb_amd.ops as ops

# rows and outputs of float_gemm.hip's tiles
TILES = [(16, 16), (32, 16), (32, 32), (48, 32), (48, 64), (48, 48), (48, 64),
         (64, 64), (80, 64), (64, 96), (80, 80)]
REFUSED = -2


def _call(tile, K, ldx):
    size = lambda n: ctypes.c_int(n)
    at = ctypes.c_void_p(4096)      # never read: there is no device
    return ops._lib.ll_float_gemm(
        at, size(4096), at, at, size(600), size(4096), size(K), size(ldx),
        size(0), size(tile), None)


@pytest.mark.skipif(torch.cuda.is_available() or not ops.native_available(),
                    reason="the addresses are none of a device")
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_offsets_of_a_tile_fit(tile):
    rows, cols = TILES[tile]
    # the first byte past the tile's last row is at offset 4 rows ld
    most_x, most_w = (2 ** 30 // n // 32 * 32 for n in (rows, cols))
    depth = min(most_x, most_w)
    assert _call(tile, 1024, most_x) != REFUSED
    assert _call(tile, 1024, most_x + 32) == REFUSED
    assert _call(tile, depth, depth) != REFUSED
    assert _call(tile, depth + 32, depth + 32) == REFUSED


def test_every_tile_is_known():
    if ops.native_available() and not torch.cuda.is_available():
        assert _call(len(TILES), 1024, 1024) == REFUSED
