"""Which products norm their rows themselves: one rule for the kernels and for
what decides before anything is allocated for them."""
import ctypes

import pytest
import torch

import llmlb_amd.ops as ops

pytestmark = pytest.mark.skipif(not ops.native_available(),
                                reason="kernels are not built")


@pytest.mark.parametrize("N, K, outputs, taken", [
    (1, 2048, 1, True), (1, 2112, 1, False), (1, 4096, 1, False),
    (1, 2048, 49152, True), (1, 2048, 49153, False),
    (1, 512, 152064, True), (1, 576, 152064, False), (2, 1024, 1, True),
    (2, 1088, 1, False), (2, 2048, 1, False), (4, 1024, 16384, True),
    (4, 1024, 16385, False), (4, 512, 32000, False), (5, 512, 1, False)])
def test_rule(N, K, outputs, taken):
    assert ops.norms_rows(torch.empty(N, K), outputs) == taken
    if torch.cuda.is_available():
        return
    # the entry refuses the same sizes, before anything of a device (which
    # there is not) is asked for
    at, i = ctypes.c_void_p(4096), ctypes.c_int
    M = outputs + -outputs % 4
    rc = ops._lib.ll_row_gemm_normed(
        at, i(M), at, at, None, None, at, ctypes.c_float(1e-5), i(N), i(M),
        i(K), i(K), i(0), i(0), None)
    assert (rc == -2) == (not taken)


def test_rows_of_other_shapes():
    assert not ops.norms_rows(torch.empty(64))
    assert not ops.norms_rows(torch.empty(1, 1, 64))
