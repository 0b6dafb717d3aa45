"""Products of many rows (tile_gemm.hip) against float products of the same
numbers, at the edges of its tiles."""
import pytest
import torch

import llmlb_amd.ops as ops
from test_row_gemm_gpu import DEV, _act, _act_bound

pytestmark = pytest.mark.gpu


def _tiled(x, w, act, out, up, a, b, monkeypatch, tile=-1):
    """The kernel at sizes at which the library would be the faster."""
    monkeypatch.setattr(ops._lib, "ll_tile_gemm_gains", lambda *sizes: 1)
    return ops._tile_gemm(x, w, act, out, up, a, b, tile)


# one tile, edges of rows and outputs, several tiles a workgroup (2100 rows
# of 9000 outputs are 324 to 2343 tiles); depths of one step, fewer than are
# fetched ahead and more; tile -1: the kernel's choice
@pytest.mark.parametrize("tile,act,a,b", [
    (0, "relu2", 0, 0), (0, "gelu", 0, 0), (0, "clamped", 1.5, 1.7),
    (1, "relu2", 0, 0), (-1, "relu2", 0, 0), (4, "gelu", 0, 0),
    (-1, "clamped", 1.5, 1.7), (-1, "gelu", 0, 0), (-1, "plain", 0, 0),
    *((t, act, 0, 0) for t in range(9) for act in ("plain", "swiglu"))])
@pytest.mark.parametrize("N,M,K", [(129, 8, 64), (256, 256, 128),
                                   (300, 1160, 192), (513, 520, 1024),
                                   (2100, 9000, 64), (2100, 9000, 448)])
def test_tile_gemm(N, M, K, tile, act, a, b, monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x = torch.randn(N, K + 16, generator=g, device=DEV).bfloat16()[:, 8:8 + K]
    up = M if act in ("swiglu", "clamped") else 0
    w = torch.randn(M + up, K, generator=g, device=DEV).mul_(
        K ** -0.5).bfloat16()
    ref, bound = _act_bound(act, x, w, up, a, b)
    wide = torch.full((N, M + 16), 7.0, device=DEV, dtype=torch.bfloat16)
    out = _tiled(x, w, act, wide[:, 8:8 + M], up, a, b, monkeypatch, tile)
    assert ((out.double() - ref).abs() <= bound).all()
    assert (wide[:, :8] == 7).all() and (wide[:, 8 + M:] == 7).all()


@pytest.mark.parametrize("act", ["gelu", "swiglu"])
def test_infinities_and_nan(act, monkeypatch):
    """What the activation of the library's product makes of them."""
    x = torch.zeros(256, 64, device=DEV, dtype=torch.bfloat16)
    x[:, 0] = 1.0
    special = torch.tensor([float("inf"), -float("inf"), float("nan"), 3e38,
                            -3e38, -90.0, 90.0, 0.0], device=DEV)
    w = torch.zeros(16, 64, device=DEV, dtype=torch.bfloat16)
    w[:, 0] = torch.cat([special, torch.ones_like(special)])
    up = 8 if act == "swiglu" else 0
    out = _tiled(x, w, act, None, up, 0, 0, monkeypatch)
    # zeros times the special numbers are in no sum: the column has one
    z = (x.float()[:, :1] * w.float()[:, 0]).bfloat16()
    ref = _act(act, z.double(), up, 0, 0)
    mine = out.double()
    assert torch.equal(mine.isnan(), ref.isnan())
    seen = ~ref.isnan()
    torch.testing.assert_close(mine[seen], ref[seen], rtol=2 ** -7,
                               atol=1e-30)


@pytest.mark.parametrize("N,M,K,shift", [(300, 12, 64, 0), (300, 64, 72, 0),
                                         (300, 64, 64, 4)])
def test_other_operands_go_to_the_library(N, M, K, shift, monkeypatch):
    x = torch.randn(N, K + 8, device=DEV).bfloat16()[:, shift:shift + K]
    w = torch.randn(M, K, device=DEV).bfloat16()
    assert _tiled(x, w, "gelu", None, 0, 0, 0, monkeypatch) is None


@torch.inference_mode()
def test_capture():
    """Replays give what an eager call gives."""
    x = torch.randn(2048, 256, device=DEV).bfloat16()
    w = torch.randn(8192, 256, device=DEV).mul_(0.06).bfloat16()
    want = ops.linear_act(x, w, "gelu")
    assert want is not None
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = ops.linear_act(x, w, "gelu")
    for i in range(3):
        x.add_(1.0)
        want = ops.linear_act(x, w, "gelu")
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i


def test_prompt_products():
    """The whole call, on both sides of the choice."""
    for N, M, K, taken in ((1355, 3216, 1024, True),
                           (1355, 2048, 7168, False)):
        x = torch.randn(N, K, device=DEV).bfloat16()
        w = torch.randn(M, K, device=DEV).mul_(K ** -0.5).bfloat16()
        assert (ops._tile_gemm(x, w) is not None) == taken
        z = x.double() @ w.double().T
        bound = z.abs() * 2.0 ** -8 + (
            x.double().abs() @ w.double().abs().T) * K * 2.0 ** -24
        assert ((ops.linear_rows(x, w).double() - z).abs() <= bound).all()


@pytest.mark.parametrize("N,M,K,taken", [
    (129, 1024, 1024, 1), (129, 3216, 1024, 1), (129, 2048, 2048, 0),
    (320, 32768, 2048, 0), (320, 32000, 2048, 1)])
def test_plain_products_taken(N, M, K, taken):
    """Few tiles of some depth and the widest are the library's."""
    assert ops._lib.ll_tile_gemm_gains(N, M, K, ops._ROW_ACTS["plain"]) \
        == taken


def test_gradients_keep_the_library():
    x = torch.randn(300, 64, device=DEV, dtype=torch.bfloat16,
                    requires_grad=True)
    w = torch.randn(512, 64, device=DEV, dtype=torch.bfloat16)
    ops.linear_rows(x, w).float().sum().backward()
    assert x.grad is not None


def _operands():
    x = torch.randn(300, 64, device=DEV).bfloat16()
    return x, torch.randn(4096, 64, device=DEV).bfloat16()


@torch.inference_mode()
def test_autocast_keeps_the_library():
    x, w = _operands()
    assert ops.linear_act(x, w, "gelu") is not None
    heads = x[:100].view(2, 50, 64), w.view(2, 2048, 64)
    with torch.autocast("cuda", torch.float16):
        assert ops.linear_rows(x, w).dtype == torch.float16
        assert ops.linear_act(x, w, "gelu") is None
        assert not ops.linear_heads(*heads, x.new_empty(2, 50, 2048))
    assert ops.linear_heads(*heads, x.new_empty(2, 50, 2048))


@torch.inference_mode()
def test_operands_of_another_device_keep_the_library(monkeypatch):
    """Kernels are launched on the current device's stream."""
    x, w = _operands()
    want = torch.nn.functional.linear(x, w)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert torch.equal(ops.linear_rows(x, w), want)
    assert ops.linear_act(x, w, "gelu") is None
    assert not ops.linear_heads(x[:100].view(2, 50, 64), w.view(2, 2048, 64),
                                x.new_empty(2, 50, 2048))
