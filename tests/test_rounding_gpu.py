"""What kernels store as bf16 is the nearest number, ties to even: the
hardware's conversion against the host's, bit by bit."""
import pytest
import torch

import llmlb_amd.ops as ops
from llmlb_amd.ops import hybrid as hy
from test_tile_gemm_gpu import _tiled

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _floats(n):
    """Every sign and exponent, with last bits at, beside and between ties:
    subnormal numbers, infinities and NaN among them."""
    g = torch.Generator().manual_seed(n)
    high = torch.arange(n) * 65536 // n
    low = torch.tensor([0, 1, 0x7FFF, 0x8000, 0x8001, 0xFFFF])
    bits = high << 16 | low[torch.randint(6, (n,), generator=g)]
    return torch.where(bits < 2 ** 31, bits, bits - 2 ** 32).int().view(
        torch.float32)


def _same(got, want):
    got, want = got.cpu(), want.cpu()
    assert torch.equal(got.isnan(), want.isnan())
    seen = ~want.isnan()
    assert torch.equal(got[seen], want[seen])


# whole vectors, and widths that are stored number by number
@pytest.mark.parametrize("width", [8, 1024, 1023])
def test_stores(width):
    x = _floats(196608 // width * width).view(-1, width)
    y = torch.zeros(x.shape, dtype=torch.bfloat16, device=DEV)
    mine, xb = x.to(DEV), torch.empty_like(y)
    hy.post_norm_add(mine, xb, y, torch.ones(width, device=DEV), 1e-5)
    _same(xb, x.bfloat16())


@pytest.mark.parametrize("act", ["plain", "relu2"])
@pytest.mark.parametrize("tile", [0, 1, 6])
def test_tile_gemm(tile, act, monkeypatch):
    """Sums of two numbers, which a float holds: the second is half a unit in
    the last place of the first, or as much and a bit."""
    g = torch.Generator().manual_seed(tile)
    first = torch.randn(1024, generator=g).bfloat16().float()
    half = torch.exp2(first.abs().log2().floor() - 8)
    more = torch.tensor([1.0, -1.0, 1.0078125, -0.9921875])
    w = torch.zeros(1024, 64)
    w[:, 0], w[:, 1] = first, half * more.repeat(256)
    x = torch.zeros(300, 64)
    x[:, :2] = 1.0
    out = _tiled(x.bfloat16().to(DEV), w.bfloat16().to(DEV), act, None, 0, 0,
                 0, monkeypatch, tile)
    want = w.sum(1).bfloat16()
    if act == "relu2":
        want = (want.float().clamp(min=0) ** 2).bfloat16()
    _same(out, want.expand(300, -1))
