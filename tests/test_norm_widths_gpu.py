"""Norms of the stream at the widths where a thread keeps one vector more."""
import pytest
import torch

from llmlb_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("width", [8, 2040, 2048, 2056, 4096, 4104, 8192])
@pytest.mark.parametrize("top", [0, 2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_add_norms(width, top, dtype):
    g = torch.Generator().manual_seed(width)
    x = torch.randn(3, width, generator=g)
    y = torch.randn(3, width, generator=g).to(dtype)
    w1, w2 = (1 + 0.3 * torch.randn(width, generator=g) for _ in range(2))
    z = torch.randn(3, 2, width, generator=g).to(dtype)
    zw = torch.rand(3, 2, generator=g)
    total = x.double() + y.double()
    if top:
        total += (z.double() * zw.double()[..., None]).sum(1)
    dev = x.to(DEV)
    h1, h2 = hy.add_norms(dev, y.to(DEV), w1.to(DEV), w2.to(DEV), 1e-5,
                          dtype, 1.0, (z.to(DEV), zw.to(DEV)) if top else None)
    # four float additions of terms below 4 max; a norm of ``width`` squares
    # is off by less than width 2^-24 of itself (its root by half), and a
    # result in 16 bits by 2^-8
    assert (dev.cpu() - total).abs().max() <= 2.0 ** -20 * total.abs().max()
    norm = total * (total.square().mean(1, keepdim=True) + 1e-5).rsqrt()
    rel = width * 2.0 ** -24 + 2.0 ** -20 \
        + (2.0 ** -8 if dtype == torch.bfloat16 else 0)
    for h, w in ((h1, w1), (h2, w2)):
        want = norm * w
        assert (h.cpu().double() - want).abs().max() <= \
            rel * want.abs().max() + 1e-6
