"""Attention of single tokens with one and two tiles of keys on their way: no
keys but one, ends of a tile, odd and even tiles, few workgroups and many."""
import pytest
import torch

from llmlb_amd.ops import hybrid as hy
from llmlb_amd.ops import reference_hybrid as ref
from test_window_layer_gpu import operands

pytestmark = pytest.mark.gpu


def plain(window, cache):
    """By the plain implementation, in float on the CPU."""
    out, proj, g_off, H, G, D, V, _, b, size, chunk = window
    for k in ("pos", "row", "block_tables"):
        setattr(b, k, getattr(b, k).cpu())
    got = torch.zeros(out.shape, dtype=torch.float32)
    ref.window_attention(got, proj.cpu(), g_off, H, G, D, V, cache, b, size,
                         chunk)
    return got


# heads of all ways: small, with keys that two workgroups read, wide, of
# unequal sides, and larger than 128
@pytest.mark.parametrize("H, G, D, V", [
    (16, 8, 64, 64), (8, 8, 24, 32), (40, 1, 64, 64), (8, 2, 128, 128),
    (40, 1, 96, 72), (16, 8, 48, 120), (4, 2, 256, 256), (40, 1, 136, 64)])
@pytest.mark.parametrize("n", [3, 34])
@pytest.mark.parametrize("ctx", [0, 63, 64, 127, 128, 191, 192, 330])
def test_tiles(H, G, D, V, n, ctx):
    args = operands(n, 16, H, G, D, V, 8, 0, 1, 1, ctx, 4096, False, seed=ctx)
    window, mid = args[0], args[6]
    hy.window_attention(*window)
    got = mid.float().cpu()
    cache = window[7].cpu().float()
    want = plain(window, cache)
    sizes = cache.view(-1, G, 16, D + V).clone()
    sizes[..., D:].abs_()
    most = plain(window, sizes.view_as(cache))
    # weights and result are rounded to 8 bits, 2^-9 each; a score's sum of
    # D float products is off by less than that
    assert ((got - want).abs() <= 2.0 ** -7 * most).all()
