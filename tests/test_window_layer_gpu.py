"""A parallel layer's independent halves in one launch each, against the
launches they replace and sums of 64 bits."""
import types

import pytest
import torch

import llmlb_amd.ops as ops
from llmlb_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
B16 = torch.bfloat16


def operands(n, W, H, G, D, V, ff, shared, E, top, ctx, size, chunk, seed=0):
    g = torch.Generator().manual_seed(seed)

    def rand(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).to(B16).to(DEV)

    g_off = H * D
    ld = g_off + H + -(g_off + H) % 8
    proj = rand(n, ld)
    pages = ctx // 16 + 1
    cache = rand(n * pages, G * 16 * (D + V))
    pos = torch.randint(0, ctx + 1, (n,), generator=g)
    pos[0] = ctx
    index = torch.stack([torch.randperm(E, generator=g)[:top]
                         for _ in range(n)])
    bt = torch.randperm(n * pages, generator=g).view(n, pages)
    row = torch.randperm(n, generator=g)
    b = types.SimpleNamespace(
        n_tok=n, n_short=n, decode=True, max_keys=ctx + 1,
        **{k: t.to(torch.int32).to(DEV)
           for k, t in (("pos", pos), ("row", row), ("block_tables", bt))})
    mid = rand(n, H * V + shared)
    window = (mid[:, :H * V], proj, g_off, H, G, D, V, cache, b, size, chunk)
    return (window, rand(n, W), index.to(torch.int32).to(DEV), None,
            rand(E, ff, W, std=W ** -0.5), rand(E, W, ff, std=ff ** -0.5),
            mid, rand(W, H * V + shared, std=0.05))


def check(args):
    window, h, index, _, w_up, w_down, mid, w_out = args
    plain = mid.clone()
    hy.window_attention(plain[:, :window[0].shape[1]], *window[1:])
    z0 = hy.experts(h, index, None, w_up, w_down)
    both = hy.few_layer(*args)
    assert both is not None
    y, z = both
    assert torch.equal(mid, plain)      # the same steps in the same order
    # one rounding to 8 bits, and K float additions in any order
    x, w = mid.double(), w_out.double()
    K = x.shape[1]
    bound = (x @ w.t()).abs() * 2 ** -8 \
        + K * 2.0 ** -24 * (x.abs() @ w.abs().t())
    assert ((y.double() - x @ w.t()).abs() <= bound).all()
    # the first product's sums may round to a neighbour, 2^-7 of each
    u = torch.einsum("tw,tkfw->tkf", h.double(),
                     w_up.double()[index.long()]).clamp(min=0) ** 2
    spread = torch.einsum("tkf,tkwf->tkw", u, w_down.double()[
        index.long()].abs())
    assert ((z.double() - z0.double()).abs()
            <= z0.double().abs() * 2 ** -7 + spread * 2 ** -7 + 1e-30).all()


# rows of one tile, two and more; one workgroup and several a sequence;
# heads that fill a tile of 16 and more
@pytest.mark.parametrize("n", [1, 15, 17, 33, 64, 128])
@pytest.mark.parametrize("H, G, D, V", [(4, 2, 64, 64), (8, 2, 128, 128),
                                        (40, 2, 40, 24), (4, 4, 104, 72)])
def test_halves(n, H, G, D, V):
    check(operands(n, 128, H, G, D, V, 64, 32, 16, 4, 200, 4096, False,
                   seed=n))


# outputs, depths and experts that are no whole tiles; many pairs an expert,
# experts without any; one, two and five tiles of outputs of the experts' own
@pytest.mark.parametrize("W, ff, shared, E, top, n", [
    (72, 40, 0, 3, 3, 40), (200, 8, 8, 64, 1, 5), (1032, 264, 72, 8, 2, 60),
    (4096, 1288, 40, 16, 4, 61), (2048, 512, 512, 2, 1, 128)])
def test_sizes(W, ff, shared, E, top, n):
    check(operands(n, W, 4, 2, 64, 64, ff, shared, E, top, 90, 64, False))


@pytest.mark.parametrize("size, chunk, ctx", [
    (64, False, 700), (1, False, 40), (48, True, 300), (4096, False, 3000)])
@pytest.mark.parametrize("n", [2, 40])
def test_masks_and_parts(size, chunk, ctx, n):
    check(operands(n, 128, 4, 1, 128, 128, 64, 32, 8, 2, ctx, size, chunk))


def test_other_routes():
    """What the halves' own kernels keep."""
    args = list(operands(4, 128, 4, 2, 64, 64, 64, 32, 8, 2, 60, 64, False))
    assert hy.few_layer(*args) is not None
    for D, V in ((32, 32), (64, 72), (136, 128), (256, 256)):
        assert hy.few_layer(*operands(4, 128, 4, 2, D, V, 64, 32, 8, 2, 60,
                                      64, False)) is None
    lists = (torch.zeros(8, device=DEV), torch.zeros(8, 4, device=DEV))
    assert hy.few_layer(*args[:3], lists, *args[4:]) is None
    assert hy.few_layer(*args[:7], args[7].float()) is None
    assert hy.few_layer(*args[:7], args[7].t().contiguous().t()) is None
    grown = args[7].clone().requires_grad_()
    assert hy.few_layer(*args[:7], grown) is None
    args[0][8].n_short = 3              # a prompt's tokens among them
    assert hy.few_layer(*args) is None


@torch.inference_mode()     # as all captures of a process
def test_captured():
    """Replays with eager work between them."""
    args = operands(20, 256, 4, 2, 64, 64, 64, 32, 8, 2, 300, 64, False)
    want = [t.clone() for t in hy.few_layer(*args)]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = hy.few_layer(*args)
    for _ in range(3):
        for t in got:
            t.zero_()
        args[6][:, :256].zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)
        ops.linear_decode(args[6], args[7])


# output products with launches of their own: deep for their width beside short
# experts, 8192 deep, and of many tiles
@pytest.mark.parametrize("W, ff, shared, E, n", [
    (72, 40, 1000, 4, 5), (128, 64, 8192, 16, 40), (4096, 64, 5632, 4, 70)])
def test_products_apart(W, ff, shared, E, n):
    check(operands(n, W, 4, 2, 64, 64, ff, shared, E, 2, 150, 64, False))


def test_large_tiles_of_experts():
    """16 pairs an expert and few keys, or 24, where their own kernel has
    tiles of 80 outputs."""
    sizes = (2048, 4, 2, 64, 64, 1040, 0, 16, 4)
    for n, ctx, size, taken in ((64, 60, 4096, False), (64, 300, 100, False),
                                (64, 300, 4096, True), (60, 60, 4096, True),
                                (95, 800, 4096, True),
                                (96, 800, 4096, False)):
        args = operands(n, *sizes, ctx, size, False)
        assert (hy.few_layer(*args) is not None) == taken
