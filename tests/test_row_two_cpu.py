"""Two products in one launch where one tile does for both: decided before
anything of the GPU is asked for."""
import ctypes

import pytest
import torch

import llmlb_amd.ops as ops


@pytest.mark.skipif(torch.cuda.is_available() or not ops.native_available(),
                    reason="the addresses are none of a device")
@pytest.mark.parametrize("N, M1, M2, K, together", [
    (1, 8192, 6144, 4096, True), (64, 8192, 6144, 4096, True),
    (72, 8192, 6144, 4096, False), (128, 8192, 6144, 4096, False),
    (128, 8192, 6144, 2048, True), (72, 6144, 4096, 6144, False),
    (64, 1024, 14336, 4096, False), (64, 1024, 14336, 1024, True),
    (16, 10240, 11904, 4096, True), (16, 16384, 5632, 6144, False),
    (64, 4160, 2176, 1024, True), (128, 16512, 11904, 4096, True)])
def test_one_tile_for_both(N, M1, M2, K, together):
    at, i, f = ctypes.c_void_p(4096), ctypes.c_int, ctypes.c_float
    rc = ops._lib.ll_row_gemm_two(
        at, i(M1), at, i(K), at, i(M1), at, i(M2), at, i(K), at, i(M2), i(4),
        i(M2), f(7), f(1), i(N), i(K), None)
    assert (rc != -2) == together
