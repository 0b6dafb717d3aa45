"""Products of 32-bit matrices that are refused before anything of the GPU is
asked for: strides and depths whose offsets in a tile do not fit 32 bits, and
sizes at which the library's are the faster."""
import ctypes

import pytest
import torch

import llmlb_amd.ops as ops

# rows and outputs of float_gemm.hip's tiles
TILES = [(16, 16), (32, 16), (32, 32), (48, 32), (48, 64), (48, 48), (48, 64),
         (64, 64), (80, 64), (64, 96), (80, 80)]
REFUSED = -2


def _call(tile, K, ldx, N=600, M=4096):
    size = lambda n: ctypes.c_int(n)
    at = ctypes.c_void_p(4096)      # never read: there is no device
    return ops._lib.ll_float_gemm(
        at, size(M), at, at, size(N), size(M), size(K), size(ldx), size(0),
        size(tile), None)


no_device = pytest.mark.skipif(
    torch.cuda.is_available() or not ops.native_available(),
    reason="the addresses are none of a device")


@no_device
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


# sizes on both sides of each line, of few rows and of many
@no_device
@pytest.mark.parametrize("N,M,K,library", [
    (64, 4096, 64, False), (65, 4096, 64, True), (128, 32000, 32, True),
    (512, 512, 96, False), (513, 4, 224, True), (128, 4096, 128, False),
    (129, 4096, 128, True), (1, 32000, 128, False), (512, 1024, 256, False),
    (513, 1024, 256, True), (4096, 1024, 256, True), (4097, 1024, 256, False),
    (1024, 1024, 512, True), (1025, 1024, 512, False),
    (600, 1024, 1024, False), (1, 1024, 4096, True), (127, 1024, 16384, True),
    (128, 1024, 4096, False), (1, 1024, 3328, False),
    (1, 4096, 18304, False)])
def test_the_faster_product(N, M, K, library):
    assert (_call(-1, K, K, N, M) == REFUSED) == library
    assert _call(0, K, K, N, M) != REFUSED
