"""Shares of a product that the norm after it adds up, against the joined
product and the norm of its rows."""
import pytest
import torch

import llmlb_amd.ops as ops
from llmlb_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rand(seed, *shape):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEV)


# a thread with no vector, one, and several; shares in whole fours and not
@pytest.mark.parametrize("width", [8, 2040, 2048, 2056, 4096, 4104, 8200])
@pytest.mark.parametrize("shares", [1, 3, 4, 5])
@pytest.mark.parametrize("T", [1, 33])
def test_norm_of_shares(width, shares, T):
    ws, x0, w = rand(1, shares, T, width), rand(2, T, width), rand(3, width)
    y = torch.zeros_like(ws[0])
    for part in ws:
        y = y + part
    y = y.bfloat16()
    got = []
    for rows in (ws, y):
        x, xb = x0.clone(), torch.empty(T, width, device=DEV,
                                        dtype=torch.bfloat16)
        hy.post_norm_add(x, xb, rows, w, 1e-5, 0.5)
        assert torch.equal(xb, x.bfloat16())
        got.append(x)
    # another order of the sum of squares: width 2^-24 of it, half of that
    # in its root, of the largest number added
    step = (got[1] - x0).abs().max()
    assert (got[0] - got[1]).abs().max() <= \
        width * 2.0 ** -24 * step + 2.0 ** -22 * got[1].abs().max()


@pytest.mark.parametrize("N, M, K", [(32, 4096, 8192), (64, 4096, 14336),
                                     (100, 2048, 8200)])
def test_shares_are_the_product(N, M, K):
    x, w = rand(4, N, K).bfloat16(), rand(5, M, K).bfloat16()
    parts = ops.linear_shares(x, w)
    assert parts.dtype == torch.float32 and parts.shape[1:] == (N, M)
    y = torch.zeros_like(parts[0])
    for part in parts:
        y = y + part
    assert torch.equal(y.bfloat16(), ops.linear_decode(x, w))


def test_other_products_are_not_in_shares():
    x, w = rand(6, 64, 4096).bfloat16(), rand(7, 4096, 4096).bfloat16()
    assert ops.linear_shares(x, w) is None
    x, w = rand(8, 16, 14336).bfloat16(), rand(9, 4096, 14336).bfloat16()
    assert ops.linear_shares(x, w) is None
    x = rand(8, 64, 14336).bfloat16()
    assert ops.linear_shares(x.float(), w.float()) is None
    assert ops.linear_shares(x, w.requires_grad_()) is None


def test_hooks_see_rows():
    """A watched or replaced feed-forward returns its rows, as others do."""
    from llmlb_amd.models.mixers import DenseFF
    ff = DenseFF(width=2048, ff=8192, dtype=torch.bfloat16, device=DEV)
    ff.load({"up": rand(10, 8192, 2048) * 2048 ** -0.5,
             "down": rand(11, 2048, 8192) * 8192 ** -0.5})
    x = rand(12, 100, 2048).bfloat16()
    want, shares = ff(x), ff.rows_or_shares(x)
    assert want.dtype == x.dtype and shares.dim() == 3
    seen = []
    hook = ff.register_forward_hook(lambda m, args, out: seen.append(out))
    assert torch.equal(ff.rows_or_shares(x), want)
    assert torch.equal(seen[0], want)
    hook.remove()
    plain = ff.forward
    ff.forward = lambda x: plain(x) * 2
    assert torch.equal(ff.rows_or_shares(x), want * 2)
