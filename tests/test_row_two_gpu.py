"""Two products in one launch (row_gemm.hip) against the two launches."""
import pytest
import torch

import llmlb_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(N, M, F, K):
    g = torch.Generator(device=DEV).manual_seed(N + M + F + K)

    def some(*shape):
        return torch.randn(*shape, generator=g, device=DEV).bfloat16()

    return (some(N, K + 8)[:, :K], some(M, K), some(N, K + 16)[:, 8:8 + K],
            some(2 * F, K))


def _close(out, x, w):
    """Float sums of K products, rounded once to bf16."""
    x, w = x.double(), w.double()
    ref = x @ w.T
    bound = ref.abs() * 2.0 ** -8 \
        + (x.abs() @ w.abs().T) * x.shape[1] * 2.0 ** -24
    assert ((out.double() - ref).abs() <= bound + 1e-30).all()


# each of the two smaller than a tile, alike, and much larger; all numbers of
# rows; depths of less than a piece and with a remainder
@pytest.mark.parametrize("M,F,K", [(4, 4, 8), (1028, 12, 264), (20, 2052, 136),
                                   (2564, 1284, 520), (4160, 2176, 72),
                                   (12300, 4100, 64)])
@pytest.mark.parametrize("N", [1, 16, 17, 40, 64, 65, 97, 128])
@pytest.mark.parametrize("act,a,b", [("swiglu", 0.0, 0.0),
                                     ("clamped", 3.0, 1.7)])
def test_as_two_launches(N, M, F, K, act, a, b):
    x, w, y, gu = _inputs(N, M, F, K)
    wide = torch.full((N, F + 12), 7.0, device=DEV).bfloat16()
    first = ops.linear_two(x, w, y, gu, act, wide[:, 4:4 + F], F, a, b)
    _close(first, x, w)
    assert (wide[:, :4] == 7).all() and (wide[:, 4 + F:] == 7).all()
    # gate and up of the sums rounded to bf16, one rounding apart
    z = y.double() @ gu.double().T
    near = (y.double().abs() @ gu.double().abs().T) * K * 2.0 ** -24
    g, u = z.chunk(2, 1)
    slack = z.abs() * 2.0 ** -8 + near
    dg, du = slack.chunk(2, 1)
    if act == "swiglu":
        gate, du_ = torch.nn.functional.silu(g), du
    else:
        g, u = g.clamp(max=a), u.clamp(-a, a) + 1.0
        gate, du_ = g * torch.sigmoid(b * g), du
    ref = gate * u
    # |d gate / d g| is below 1.2 for any sharpness up to 1.7
    bound = 1.2 * dg * (u.abs() + du_) + gate.abs() * du_ \
        + ref.abs() * 2.0 ** -7 + 1e-6
    assert ((wide[:, 4:4 + F].double() - ref).abs() <= bound).all()


def test_other_operands_take_two_launches():
    x, w, y, gu = _inputs(5, 64, 32, 64)
    out = torch.empty(5, 32, device=DEV).bfloat16()

    def go(x=x, w=w, y=y, gu=gu, act="clamped", out=out):
        return ops.linear_two(x, w, y, gu, act, out, 32, 3.0, 1.7)

    assert go() is not None
    assert go(act="gelu") is None
    assert go(y=y[:4]) is None                          # other rows
    assert go(x=x[:, :56], w=w[:, :56].contiguous()) is None
    assert go(x=x.float(), w=w.float()) is None
    assert go(out=out.float()) is None
    assert go(w=w[:63]) is None                         # outputs by fours
    wide = torch.randn(129, 64, device=DEV).bfloat16()
    assert ops.linear_two(wide, w, wide, gu, "clamped",
                          torch.empty(129, 32, device=DEV).bfloat16(), 32,
                          3.0, 1.7) is None
