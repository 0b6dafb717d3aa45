"""Products of few rows with a weight matrix (row_gemm.hip) against float
products of the same numbers, at the edges of its tiles."""
import pytest
import torch

import llmlb_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _close(out, x, w):
    """Float sums of K products, rounded once to bf16: half a unit in the
    last place (2^-9), and K float roundings of the sum of magnitudes."""
    x, w = x.double(), w.double()
    ref = x @ w.T
    bound = ref.abs() * 2.0 ** -8 \
        + (x.abs() @ w.abs().T) * x.shape[1] * 2.0 ** -24
    assert ((out.double() - ref).abs() <= bound + 1e-30).all()


# rows: every number of 16-row tiles and shares; depths: under one piece, a
# remainder, more pieces than waves; outputs: a remainder of every tile
@pytest.mark.parametrize("M,K", [(4, 8), (20, 72), (1036, 1024),
                                 (5644, 200), (12300, 1096), (520, 4160)])
@pytest.mark.parametrize("N", [1, 16, 17, 33, 48, 49, 64, 80, 96, 113, 128])
def test_row_gemm(N, M, K):
    g = torch.Generator(device=DEV).manual_seed(N * 7 + M + K)
    wide = torch.randn(N, K + 16, generator=g, device=DEV).bfloat16()
    w = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    x = wide[:, 8:8 + K]                       # rows of a wider matrix
    out = ops._row_gemm(x, w)
    assert out is not None and out.shape == (N, M)
    _close(out, x, w)
    assert torch.equal(out, ops.linear_decode(x, w))


@pytest.mark.parametrize("N,M,K,shift", [(3, 6, 64, 0), (3, 64, 60, 0),
                                         (3, 64, 64, 1), (3, 64, 64, 4)])
def test_other_operands_go_to_the_library(N, M, K, shift):
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(N, K + 8, generator=g, device=DEV).bfloat16()
    x = x[:, shift:shift + K]
    w = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    assert ops._row_gemm(x, w) is None
    _close(ops.linear_decode(x, w), x, w)


def test_gradients_keep_the_library():
    x = torch.randn(5, 64, device=DEV, dtype=torch.bfloat16,
                    requires_grad=True)
    w = torch.randn(32, 64, device=DEV, dtype=torch.bfloat16)
    ops.linear_decode(x, w).float().sum().backward()
    assert x.grad is not None
