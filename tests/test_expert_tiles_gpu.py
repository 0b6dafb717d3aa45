"""Products of experts' lists by tiles of 192 x 256, several of them a
workgroup, whose results are stored while the next tile is computed: against
those of 128 x 128, which make the same sums, and against float64."""
import pytest
import torch

from llmlb_amd.ops import _ptr, _stream
from llmlb_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
E, TOP = 12, 4


def _lists(T):
    """Experts with no pair, one, an edge of a tile and beside it, many."""
    sizes = [0, 1, 192, 191, 193, 384, 577, 0]
    sizes += [T, T - 1, T - 500]
    sizes.append(T * TOP - sum(sizes))
    assert max(sizes) <= T and len(sizes) == E
    order = torch.randperm(T * TOP, generator=torch.Generator().manual_seed(T))
    pairs, first = torch.zeros(E, T, dtype=torch.int32), 0
    for e, n in enumerate(sizes):
        pairs[e, :n] = order[first:first + n]
        first += n
    return torch.tensor(sizes, dtype=torch.int32).to(DEV), pairs.to(DEV)


# depths of one step, whose results are stored at once, of fewer steps than a
# tile's held stores take, as many and more; outputs that are no whole tiles
@pytest.mark.parametrize("act, div", [(1, TOP), (0, 1)])
@pytest.mark.parametrize("N", [1024, 1544])
@pytest.mark.parametrize("K", [64, 128, 192, 320, 384, 448, 1024])
def test_tiles(K, N, act, div):
    T = 5000
    counts, pairs = _lists(T)
    g = torch.Generator(device=DEV).manual_seed(K + N)
    x = torch.randn(T * TOP // div, K, generator=g, device=DEV).bfloat16()
    w = torch.randn(E, N, K, generator=g, device=DEV).mul_(
        K ** -0.5).bfloat16()

    def run(tile):
        out = torch.full((T * TOP, N), 7.0, device=DEV, dtype=torch.bfloat16)
        assert hy.native().hy_expert_tiles(
            _ptr(out), _ptr(x), _ptr(w), _ptr(counts), _ptr(pairs), hy._i(E),
            hy._i(N), hy._i(K), hy._i(div), hy._i(act), hy._i(T),
            hy._i(T * TOP), hy._i(tile), _stream()) == 0
        return out

    out = run(3)
    assert torch.equal(out, run(0))
    for e in (1, 2, 4, 8):
        rows = pairs[e, :counts[e]].long()
        want = x[rows // div].double() @ w[e].double().T
        # K additions, each off by 2^-24 of the sum of absolute products at
        # most; the square doubles an error; rounded to 8 bits
        off = K * 2.0 ** -24 * (x[rows // div].double().abs()
                                @ w[e].double().abs().T)
        if act:
            want = want.clamp(min=0)
            want, off = want ** 2, 2 * want * off + off ** 2
        bound = off + 2.0 ** -8 * (want.abs() + off)
        assert ((out[rows].double() - want).abs() <= bound).all()


# ten tiles a workgroup: more than the lists in LDS have places
@pytest.mark.parametrize("K", [64, 128, 192, 256])
def test_many_tiles(K):
    T, N, act, div = 16384, 1544, 1, TOP
    counts, pairs = _lists(T)
    g = torch.Generator(device=DEV).manual_seed(K)
    x = torch.randn(T, K, generator=g, device=DEV).bfloat16()
    w = torch.randn(E, N, K, generator=g, device=DEV).mul_(
        K ** -0.5).bfloat16()
    outs = []
    for tile in (3, 0):
        out = torch.full((T * TOP, N), 7.0, device=DEV, dtype=torch.bfloat16)
        assert hy.native().hy_expert_tiles(
            _ptr(out), _ptr(x), _ptr(w), _ptr(counts), _ptr(pairs), hy._i(E),
            hy._i(N), hy._i(K), hy._i(div), hy._i(act), hy._i(T),
            hy._i(T * TOP), hy._i(tile), _stream()) == 0
        outs.append(out)
    assert torch.equal(*outs)
