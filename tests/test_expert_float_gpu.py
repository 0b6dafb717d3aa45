"""Experts' products in 32 bits (experts.hip) against 64-bit products of the same
numbers, at the edges of their tiles."""
import pytest
import torch

from llmlb_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def run(h, index, up, down):
    """Both products of every pair, each of the numbers that it was given."""
    T, top = index.shape
    E = up.shape[0]
    flat = index.flatten()
    counts = torch.bincount(flat, minlength=E).int()
    pairs = torch.zeros(E, T, dtype=torch.int32, device=DEV)
    for e in range(E):
        mine = (flat == e).nonzero().flatten().int()
        pairs[e, :len(mine)] = mine
    z = hy.experts(h, index.int(), (counts, pairs), up, down)
    return flat, z.flatten(0, 1)


def act(u):
    return u.clamp(min=0.0).square()


# experts, choices, tokens, width, ff, how many experts are chosen from: every
# tile, whole and not, experts with no pair, one and many; depths that are whole
# pieces and (20, 36) not
@pytest.mark.parametrize("E, top, T, W, F, used", [
    (1, 1, 1, 32, 4, 1), (3, 2, 5, 1024, 36, 3), (16, 4, 9, 1024, 256, 16),
    (16, 4, 90, 1024, 256, 12), (16, 4, 130, 1024, 260, 16),
    (16, 4, 250, 544, 256, 16), (5, 1, 333, 1024, 64, 5),
    (16, 4, 700, 1024, 320, 9), (2, 2, 500, 512, 100, 2), (4, 3, 40, 20, 36, 4),
    (300, 3, 70, 64, 32, 290)])
def test_experts(E, top, T, W, F, used):
    g = torch.Generator(device=DEV).manual_seed(E + T)
    h = torch.randn(T, W, generator=g, device=DEV)
    up = torch.randn(E, F, W, generator=g, device=DEV) * W ** -0.5
    down = torch.randn(E, W, F, generator=g, device=DEV) * F ** -0.5
    index = torch.rand(T, used, generator=g, device=DEV).argsort(1)[:, :top]
    flat, z = run(h, index.contiguous(), up, down)
    for e in flat.unique().tolist():
        p = (flat == e).nonzero().flatten()
        x, a, b = h[p // top].double(), up[e].double(), down[e].double()
        s = x @ a.T
        # of every product 2^-24 is left out at most, and a sum of n is rounded
        # less than n times; the square doubles what the first has lost
        off = (x.abs() @ a.abs().T) * (W + 1) * 2.0 ** -24
        u = act(s)
        lost = 2 * off * (s.clamp(min=0.0) + off) + 2.0 ** -23 * u
        bound = lost @ b.abs().T + (u + lost) @ b.abs().T * (
            (F + 1) * 2.0 ** -24)
        assert ((z[p].double() - u @ b.T).abs() <= bound).all()
        # and on the whole no more than sums in 32 bits are
        assert (z[p].double() - u @ b.T).norm() <= 2e-6 * (u @ b.T).norm()


def test_numbers_that_do_not_come_apart():
    """Infinities and numbers that parts of 16 bits do not hold: results are made
    again by float instructions, those of some rows beside them as well, which
    come out as close."""
    g = torch.Generator(device=DEV).manual_seed(1)
    h = torch.randn(60, 256, generator=g, device=DEV)
    up = torch.randn(4, 64, 256, generator=g, device=DEV) / 16
    down = torch.randn(4, 256, 64, generator=g, device=DEV) / 8
    index = torch.rand(60, 4, generator=g, device=DEV).argsort(1)[:, :2]
    _, plain = run(h, index.contiguous(), up, down)
    odd = h.clone()
    odd[3, 7] = float("inf")
    odd[9] *= 1e-17                 # parts of the squares are below 2^-126
    odd[20] = 0.0
    flat, z = run(odd, index.contiguous(), up, down)
    others = torch.ones(120, dtype=torch.bool, device=DEV)
    for t in (3, 9, 20):
        others[2 * t:2 * t + 2] = False
    # either is within 2e-6 of the same, as above
    assert (z - plain)[others].norm() <= 4e-6 * plain[others].norm()
    assert not z[6:8].isfinite().all()
    assert (z[40:42] == 0).all()
    for p in (18, 19):
        e = int(flat[p])
        want = act(odd[9].double() @ up[e].double().T) @ down[e].double().T
        assert (z[p].double() - want).norm() <= 1e-5 * want.norm()


# rows that are whole vectors of four and not, at addresses that are and are not
@pytest.mark.parametrize("W, dtype", [
    (64, torch.float32), (1024, torch.float32), (1026, torch.float32),
    (1028, torch.bfloat16), (1026, torch.bfloat16)])
@pytest.mark.parametrize("at_h, at_w", [(0, 0), (1, 0), (0, 1), (2, 4)])
def test_router_at_any_address(W, dtype, at_h, at_w):
    g = torch.Generator(device=DEV).manual_seed(W)
    T, E = 21, 13
    flat_h = torch.randn(T * W + 8, generator=g, device=DEV).to(dtype)
    flat_w = (torch.randn(E * W + 8, generator=g, device=DEV)
              * 3.0 * W ** -0.5).to(dtype)
    h = flat_h[at_h:at_h + T * W].view(T, W)
    w = flat_w[at_w:at_w + E * W].view(E, W)
    index, weight, _ = hy.route(h, w, E, 1, 1, 1.0, False)
    want = (h.double() @ w.double().T).softmax(1)
    got = torch.zeros(T, E, dtype=torch.float64, device=DEV)
    got.scatter_(1, index.long(), weight.double())
    # a logit is off by W 2^-24 of its products' sizes at most, and so is the
    # logarithm of a share of all by twice that and a few roundings more
    off = W * 2.0 ** -24 * (h.double().abs() @ w.double().abs().T).max()
    assert (got - want).abs().max() <= 2 * off + 2.0 ** -20
