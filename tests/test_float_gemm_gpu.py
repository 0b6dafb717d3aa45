"""Products of 32-bit matrices (float_gemm.hip) against 64-bit products of the
same numbers, at the edges of its tiles."""
import pytest
import torch

import llmlb_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TILES = 11


def _close(out, x, w):
    """Of every product 2^-24 is left out at most, and a sum of K is rounded
    less than K times."""
    x, w = x.double(), w.double()
    bound = (x.abs() @ w.abs().T) * (x.shape[1] + 1) * 2.0 ** -24
    assert ((out.double() - x @ w.T).abs() <= bound).all()


def _rows(N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(N, K + 8, generator=g, device=DEV)[:, 4:4 + K]


# depths of one piece, of fewer pieces than waves and of a remainder; rows and
# outputs that are no whole tiles; matrices narrow enough to go by rows
@pytest.mark.parametrize("tile", range(TILES))
@pytest.mark.parametrize("N,M,K", [
    (1, 4, 32), (17, 36, 160), (50, 68, 288), (65, 260, 1056), (81, 100, 128),
    (1030, 100, 64), (300, 1028, 96), (700, 2052, 32)])
def test_tiles(N, M, K, tile):
    x, w = _rows(N, K, N + M), _rows(M, K, K).contiguous()
    wide = torch.full((N, M + 8), 7.0, device=DEV)
    out = ops._float_gemm(x, w, out=wide[:, 4:4 + M], tile=tile)
    _close(out, x, w)
    assert (wide[:, :4] == 7).all() and (wide[:, 4 + M:] == 7).all()


@pytest.mark.parametrize("N,M,K", [(1, 1024, 1024), (300, 288, 1024),
                                   (600, 1024, 3328)])
def test_errors_are_not_the_librarys(N, M, K):
    x, w = _rows(N, K, 1), _rows(M, K, 2).contiguous()
    ref = x.double() @ w.double().T
    ours, library = ((t.double() - ref).norm() / ref.norm() for t in
                     (ops.linear_rows(x, w), torch.nn.functional.linear(x, w)))
    assert ours <= library


@pytest.mark.parametrize("act", ["relu2", "gelu"])
@pytest.mark.parametrize("N", [5, 130])
def test_activations_are_those_of_their_own_kernels(N, act):
    from llmlb_amd.ops import hybrid as hy
    x, w = _rows(N, 256, 3), _rows(512, 256, 4).contiguous()
    z = ops._float_gemm(x, w)
    if act == "gelu":
        hy.gelu_tanh_(z)
    else:
        hy.squared_relu(z, z)
    assert torch.equal(ops.linear_act(x, w, act), z)


def test_numbers_that_do_not_come_apart():
    """Infinities, no numbers, numbers that round up to infinity as bf16, and
    ones whose parts bf16 does not hold."""
    x, w = _rows(70, 256, 5).contiguous(), _rows(68, 256, 6).contiguous()
    inf = float("inf")
    x[3, 7], x[5, 9], w[11, 3] = inf, float("nan"), -inf
    x[8], x[20, 5] = 3e38 / 256, 3.402e38
    w[30] *= 1e-30
    x[40] *= 1e-36
    x[41] = 0.0
    out, ref = ops.linear_rows(x, w), (x.double() @ w.double().T)
    exact = ref.float()
    assert torch.equal(out.isnan(), exact.isnan())
    assert torch.equal(out.isinf(), exact.isinf())
    assert torch.equal(out[out.isinf()], exact[exact.isinf()])
    keep = [i for i in range(70) if i not in (3, 5, 20)]
    cols = [i for i in range(68) if i != 11]
    x, w, out = x[keep], w[cols], out[keep][:, cols]
    # what is below the smallest normal number may be lost
    bound = (x.double().abs() @ w.double().abs().T) \
        * (2.0 ** -21 + 256 * 2.0 ** -24) + 256 * 2.0 ** -126
    assert ((out.double() - x.double() @ w.double().T).abs() <= bound).all()


@pytest.mark.parametrize("N,M,K,shift", [(3, 6, 64, 0), (3, 64, 48, 0),
                                         (3, 64, 64, 1), (513, 64, 224, 0)])
def test_other_operands_go_to_the_library(N, M, K, shift):
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(N, K + 4, generator=g, device=DEV)[:, shift:shift + K]
    w = torch.randn(M, K, generator=g, device=DEV)
    assert ops._float_gemm(x, w) is None
    assert torch.equal(ops.linear_rows(x, w),
                       torch.nn.functional.linear(x, w))
    assert torch.equal(ops.linear_decode(x, w),
                       torch.nn.functional.linear(x, w))


def test_gradients_and_autocast_keep_the_library():
    x = torch.randn(5, 64, device=DEV, requires_grad=True)
    w = torch.randn(32, 64, device=DEV)
    ops.linear_rows(x, w).sum().backward()
    assert x.grad is not None
    x = x.detach()
    with torch.autocast("cuda", torch.bfloat16):
        assert ops.linear_rows(x, w).dtype == torch.bfloat16
        assert ops.linear_act(x, w, "gelu") is None


@torch.inference_mode()     # as all captures of a process
def test_captured():
    x, w = _rows(300, 512, 8).contiguous(), _rows(640, 512, 9).contiguous()
    graph = torch.cuda.CUDAGraph()
    ops.linear_rows(x, w)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = ops.linear_rows(x, w)
    for seed in range(3):
        x.copy_(_rows(300, 512, seed))
        graph.replay()
        assert torch.equal(out, ops.linear_rows(x, w))


@pytest.mark.parametrize("tile", [-1, 7, 8, 10])
def test_long_strides(tile):
    """Rows 14 million numbers apart: past 32 bits in tiles of 80 rows."""
    x = torch.zeros(97, 14_000_000, device=DEV)[:, :64]
    x.copy_(_rows(97, 64, 12))
    w = _rows(4096, 64, 13).contiguous()
    out = ops._float_gemm(x, w, tile=tile)
    assert (out is None) if tile >= 8 else (tile < 0 or out is not None)
    _close(ops.linear_rows(x, w) if out is None else out, x, w)


@pytest.mark.parametrize("K", [32, 96, 256])
def test_shallow_errors_are_not_the_librarys(K):
    g = torch.Generator(device=DEV).manual_seed(K)
    near = [1 + 0.01 * torch.rand(300, K, generator=g, device=DEV)
            for _ in range(2)]
    for x, w in ((_rows(300, K, 1), _rows(256, K, 2).contiguous()),
                 (near[0], near[1][:256].contiguous())):
        ref = x.double() @ w.double().T
        off = [t.double() - ref for t in
               (ops._float_gemm(x, w), torch.nn.functional.linear(x, w))]
        assert off[0].norm() <= off[1].norm()
    # what is left out of these has the sign of the parts: to either side, so
    # that 76800 sums average far below a float's last bit
    assert abs((off[0] / ref).mean()) < 2.0 ** -27


def test_rows_of_one_number():
    """2^-24 are left out at most, and the last of the parts' sums may be cut
    off, not rounded: 2^-23."""
    x = torch.zeros(256, 128, device=DEV)
    x[torch.arange(256), torch.arange(256) % 128] = _rows(256, 32, 14)[:, 0]
    w = _rows(512, 128, 15).contiguous()
    ref = x.double() @ w.double().T
    off = ((ops._float_gemm(x, w).double() - ref) / ref).abs()
    assert off.max() <= 1.5 * 2.0 ** -23


# numbers of which bf16 parts are too small, or nothing is left, by numbers
# large enough to tell (of 288 normal numbers times 3e36 by ordinary ones sums
# stay below infinity to 6 times their spread); both ways round, and results that
# are small themselves
@pytest.mark.parametrize("of_x,of_w", [
    (1e-36, 1e30), (1e30, 1e-36), (1e-39, 1e30), (1e-42, 3e36), (1e-33, 1e5),
    (1e-30, 1.0), (1.0, 1e-37), (1e-20, 1e-16), (1e-39, 1.0), (1e-25, 1e25),
    (3e38 / 256, 1.0)])
@pytest.mark.parametrize("tile", [-1, 0, 4, 8, 9])
def test_small_by_large_numbers(of_x, of_w, tile):
    x, w = _rows(70, 288, 16) * of_x, _rows(68, 288, 17) * of_w
    # beside an ordinary row and output, one of a single number and of none
    x[5], w[9] = _rows(1, 288, 18)[0], _rows(1, 288, 19)[0]
    x[33, 1:], w[20], x[64] = 0, 0, 0
    out = ops._float_gemm(x, w.contiguous(), tile=tile).double()
    x, w = x.double(), w.double()
    bound = (x.abs() @ w.abs().T) * (288 * 2.0 ** -24 + 2.0 ** -22) \
        + 288 * 2.0 ** -149
    assert ((out - x @ w.T).abs() <= bound).all()
    assert (out[64] == 0).all() and (out[:, 20] == 0).all()


@pytest.mark.parametrize("tile", range(TILES))
def test_outputs_made_again(tile):
    """Blocks of 16 x 16 of a tile's edges and middle, and activations of
    them."""
    x, w = _rows(175, 160, 20).contiguous(), _rows(200, 160, 21).contiguous()
    for r in (0, 47, 95, 174):
        x[r] *= 1e-30
    x[100, 3], w[150, 2] = float("inf"), float("nan")
    ref = x.double() @ w.double().T
    out = ops._float_gemm(x, w, tile=tile)
    assert torch.equal(out.isnan(), ref.isnan())
    assert torch.equal(out[100].isinf(), ref[100].isinf())
    keep = torch.tensor([r for r in range(175) if r != 100], device=DEV)
    cols = torch.tensor([c for c in range(200) if c != 150], device=DEV)
    _close(out[keep][:, cols], x[keep], w[cols])
    assert torch.equal(ops._float_gemm(x, w, "relu2", tile=tile)[keep][:, cols],
                       out[keep][:, cols].clamp(min=0) ** 2)
