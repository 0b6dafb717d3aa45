"""Where a parallel layer's output product and its experts' second product are
launches of their own: decided before anything of the GPU is asked for."""
import ctypes

import pytest
import torch

from llmlb_amd.ops import hybrid as hy

APART = 0


@pytest.mark.skipif(torch.cuda.is_available()
                    or not hy.library_path("hybrid").exists(),
                    reason="the addresses are none of a device")
@pytest.mark.parametrize("N, M, K, E, F, apart", [
    # both sides of each line: depth to outputs with short experts, 8192 deep,
    # tiles, tiles times depth
    (1, 1024, 3072, 16, 256, False), (1, 1024, 3080, 16, 256, True),
    (1, 1024, 4096, 64, 256, False), (32, 4096, 12288, 16, 1280, False),
    (33, 4096, 8184, 64, 1280, True), (33, 2048, 5376, 16, 512, False),
    (33, 2048, 8192, 64, 512, True), (61, 4096, 5376, 16, 1280, False),
    (65, 4096, 5376, 16, 1280, True), (96, 8160, 512, 8, 1536, False),
    (96, 8192, 512, 8, 1536, True), (128, 2048, 5376, 16, 512, False)])
def test_line(N, M, K, E, F, apart):
    lib = ctypes.CDLL(str(hy.library_path("hybrid")))
    at, i = ctypes.c_void_p(4096), ctypes.c_int
    done = lib.hy_down_out(at, at, at, i(N), i(M), i(K), at, at, at, at,
                           i(E), i(M), i(F), i(4 * N), None)
    assert (done == APART) == apart and done <= APART
