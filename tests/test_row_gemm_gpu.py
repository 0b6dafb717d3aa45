"""Products of few rows with a weight matrix (row_gemm.hip) against float
products of the same numbers, at the edges of its tiles."""
import pytest
import torch

import llmlb_amd.ops as ops
from llmlb_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _close(out, x, w):
    """Float sums of K products, rounded once to bf16: half a unit in the
    last place (2^-9), and K float roundings of the sum of magnitudes."""
    x, w = x.double(), w.double()
    ref = x @ w.T
    bound = ref.abs() * 2.0 ** -8 \
        + (x.abs() @ w.abs().T) * x.shape[1] * 2.0 ** -24
    assert ((out.double() - ref).abs() <= bound + 1e-30).all()


# rows: every number of 16-row tiles and shares; depths: under one piece, a
# remainder, more pieces than waves; outputs: a remainder of every tile
@pytest.mark.parametrize("M,K", [(4, 8), (20, 72), (1036, 1024),
                                 (5644, 200), (12300, 1096), (520, 4160)])
@pytest.mark.parametrize("N", [1, 16, 17, 33, 48, 49, 64, 80, 96, 97, 113, 128])
def test_row_gemm(N, M, K):
    g = torch.Generator(device=DEV).manual_seed(N * 7 + M + K)
    wide = torch.randn(N, K + 16, generator=g, device=DEV).bfloat16()
    w = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    x = wide[:, 8:8 + K]                       # rows of a wider matrix
    out = ops._row_gemm(x, w)
    assert out is not None and out.shape == (N, M)
    _close(out, x, w)
    assert torch.equal(out, ops.linear_decode(x, w))


# rows and outputs at which each tile is taken (of 16 to 64 rows of x and 16
# to 112 of W), with remainders
@pytest.mark.parametrize("N,M", [
    (1, 4), (1, 1028), (1, 12332), (76, 1284), (1, 8196), (1, 11924),
    (1, 16412), (106, 516), (106, 1028), (106, 2564), (31, 12332),
    (31, 16412), (31, 20492), (106, 2052), (76, 4100), (76, 6148), (76, 8196), (76, 10292),
    (106, 3076), (106, 4100), (106, 6148), (106, 8196), (106, 10292),
    (31, 24708), (76, 12332), (106, 12332)])
@pytest.mark.parametrize("K", [72, 520])
def test_tiles(N, M, K):
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x = torch.randn(N, K, generator=g, device=DEV).bfloat16()
    w = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    _close(ops._row_gemm(x, w), x, w)
    # gate and up are half as many outputs of as many rows
    if M > 4:
        test_row_gemm_with_activation(N, (M + 4) // 8 * 4, K, "swiglu", 0, 0)


# two to six shares, depths and rows that are no whole pieces or tiles
@pytest.mark.parametrize("M,K", [(4096, 8200), (2564, 12296), (1348, 17000)])
@pytest.mark.parametrize("N", [32, 41, 64, 100, 128])
def test_row_gemm_in_shares(N, M, K):
    assert ops._require_native().ll_row_gemm_shares(N, M, K) > 1
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x = torch.randn(N, K, generator=g, device=DEV).bfloat16()
    w = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    wide = torch.full((N, M + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    out = ops._row_gemm(x, w, out=wide[:, 4:4 + M])
    _close(out, x, w)
    assert (wide[:, :4] == 7).all() and (wide[:, 4 + M:] == 7).all()


@pytest.mark.parametrize("N,M,K,shift", [(3, 6, 64, 0), (3, 64, 60, 0),
                                         (3, 64, 64, 1), (3, 64, 64, 4)])
def test_other_operands_go_to_the_library(N, M, K, shift):
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(N, K + 8, generator=g, device=DEV).bfloat16()
    x = x[:, shift:shift + K]
    w = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    assert ops._row_gemm(x, w) is None
    _close(ops.linear_decode(x, w), x, w)


def test_largest_matrices_of_many_rows_go_to_the_library():
    w = torch.randn(98336, 4096, device=DEV, dtype=torch.bfloat16)
    x = torch.randn(65, 4096, device=DEV, dtype=torch.bfloat16)
    assert ops._row_gemm(x, w) is None
    assert ops._row_gemm(x, w, "swiglu", up=49168) is None
    assert ops._row_gemm(x[:64], w) is not None
    assert ops._row_gemm(x, w[:98304]) is not None
    assert torch.equal(ops.linear_decode(x, w),
                       torch.nn.functional.linear(x, w))


def test_gradients_keep_the_library():
    x = torch.randn(5, 64, device=DEV, dtype=torch.bfloat16,
                    requires_grad=True)
    w = torch.randn(32, 64, device=DEV, dtype=torch.bfloat16)
    ops.linear_decode(x, w).float().sum().backward()
    assert x.grad is not None


def _act(act, z, up, a, b):
    if act == "relu2":
        return z.clamp(min=0.0).square()
    if act == "gelu":
        return torch.nn.functional.gelu(z, approximate="tanh")
    if act == "capped":
        return a * torch.tanh(z / a) if a else z
    g, u = z[:, :up], z[:, up:]
    if act == "swiglu":
        return torch.nn.functional.silu(g) * u
    g, u = g.clamp(max=a), u.clamp(-a, a)
    return g * torch.sigmoid(b * g) * (u + 1.0)


def _act_bound(act, x, w, up, a, b):
    """(activation of the products, how far a result may be from it).  A sum
    is K float roundings off and then a bf16 number, so it is one between two
    that are mostly neighbours; the result is between the activations of
    those (which are monotone where there are more), whose own functions are
    good to 2^-20, and rounded."""
    x, w = x.double(), w.double()
    z = x @ w.T
    off = (x.abs() @ w.abs().T) * x.shape[1] * 2.0 ** -24
    if act == "plain":
        return z, off + z.abs() * 2.0 ** -8 + 1e-30
    ref = _act(act, z.bfloat16().double(), up, a, b)
    ends = [(z + s * off).bfloat16().double() for s in (-1, 1)]
    far = torch.zeros_like(ref)
    for g in ends:
        for u in ends if up else ends[:1]:
            end = torch.cat([g[:, :up], u[:, up:]], 1) if up else g
            far = torch.maximum(far, (_act(act, end, up, a, b) - ref).abs())
    unit = 2.0 ** -20 + (0.0 if act == "capped" else 2.0 ** -8)
    return ref, far + (ref.abs() + far) * unit + 1e-30


@pytest.mark.parametrize("act,a,b", [("relu2", 0, 0), ("gelu", 0, 0),
                                     ("capped", 0, 0), ("capped", 3.0, 0),
                                     ("swiglu", 0, 0), ("clamped", 1.5, 1.7)])
@pytest.mark.parametrize("M,K", [(8, 72), (2180, 1024), (6148, 328)])
@pytest.mark.parametrize("N", [1, 23, 40, 64, 97])
def test_row_gemm_with_activation(N, M, K, act, a, b):
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x = torch.randn(N, K, generator=g, device=DEV).bfloat16()
    up = M if act in ("swiglu", "clamped") else 0
    w = torch.randn(M + up, K, generator=g, device=DEV).mul_(
        K ** -0.5).bfloat16()
    ref, bound = _act_bound(act, x, w, up, a, b)
    wide = torch.full((N, M + 16), 7.0, device=DEV, dtype=torch.bfloat16)
    out = None if act == "capped" else wide[:, 8:8 + M]
    out = ops.linear_act(x, w, act, out, up, a, b)
    if act == "capped":
        assert out.dtype == torch.float32
    else:
        assert (wide[:, :8] == 7).all() and (wide[:, 8 + M:] == 7).all()
    assert ((out.double() - ref).abs() <= bound).all()


# of few rows and of many
@pytest.mark.parametrize("act", ["gelu", "swiglu", "clamped"])
@pytest.mark.parametrize("N", [16, 130])
def test_activations_are_those_of_their_own_kernels(N, act):
    """To the bit, of every finite gate beside N numbers: divisions are a
    float's, and what underflows is what does there."""
    z = torch.arange(65536, device=DEV, dtype=torch.int32).to(
        torch.uint16).view(torch.bfloat16)
    z = z[z.isfinite()]
    M = z.numel()
    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.zeros(N, 64, device=DEV, dtype=torch.bfloat16)
    x[:, 5] = 1.0
    x[:, 6] = torch.randn(N, generator=g, device=DEV).mul_(3.0)
    w = torch.zeros(M if act == "gelu" else 2 * M, 64, device=DEV,
                    dtype=torch.bfloat16)
    w[:M, 5] = z
    w[M:, 6] = 1.0
    if act == "gelu":
        want = hy.gelu_tanh_(z.repeat(N, 1))
    else:
        both = torch.cat([z.repeat(N, 1), x[:, 6:7].expand(N, M)], 1)
        want = torch.empty(N, M, device=DEV, dtype=torch.bfloat16)
        if act == "swiglu":
            want = ops.swiglu(both)
        else:
            hy.clamped_swiglu(want, both, M, 7.0, 1.702)
    out = ops.linear_act(x, w, act, None, 0 if act == "gelu" else M, 7.0,
                         1.702)
    assert torch.equal(out, want)


# heads, outputs, depth: one and two pieces of the depth, remainders of both
@pytest.mark.parametrize("H,M,K", [(4, 512, 128), (3, 68, 72), (5, 128, 512),
                                   (2, 36, 264)])
@pytest.mark.parametrize("N", [1, 16, 48, 49, 65, 128])
@pytest.mark.parametrize("gated", [False, True])
def test_heads(N, H, M, K, gated):
    g = torch.Generator(device=DEV).manual_seed(N + M)
    wide = torch.randn(N, H * (K + 8) + 24, generator=g, device=DEV).bfloat16()
    x = wide[:, 16:16 + H * (K + 8)].unflatten(1, (H, K + 8))[..., :K] \
        .transpose(0, 1)
    w = torch.randn(H, M, K, generator=g, device=DEV).mul_(
        K ** -0.5).bfloat16()
    rows = torch.full((N, H * M + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    gate = torch.randn(N, H * M + 4, generator=g, device=DEV).bfloat16()
    gate = gate[:, 4:] if gated else None
    out = rows[:, 4:4 + H * M].unflatten(1, (H, M)).transpose(0, 1)
    assert ops.linear_heads(x, w, out, gate)
    assert (rows[:, :4] == 7).all() and (rows[:, 4 + H * M:] == 7).all()
    if not gated:
        for h in range(H):
            _close(out[h], x[h], w[h])
        return
    # a sum that may round either way, then the gate, then a rounding
    z = x.double() @ w.double().transpose(1, 2)
    ref = z * gate.double().sigmoid().view(N, H, M).transpose(0, 1)
    bound = z.abs() * 2.0 ** -7 \
        + (x.double().abs() @ w.double().abs().transpose(1, 2)) * K * 2.0 ** -24
    assert ((out.double() - ref).abs() <= bound).all()


# columns of W: one and two pieces of the depth, remainders of both; from
# 8192 outputs of all heads on 64 a tile, past 1024 workgroups of 32 rows
@pytest.mark.parametrize("H,K,M", [(4, 128, 512), (3, 72, 72), (5, 512, 136),
                                   (2, 8, 8), (2, 264, 40), (16, 72, 520),
                                   (17, 264, 520)])
@pytest.mark.parametrize("N", [1, 16, 48, 49, 65, 128])
def test_heads_against_columns(N, H, K, M):
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x = torch.randn(N, H, K + 8, generator=g, device=DEV).bfloat16()[
        ..., 8:].transpose(0, 1)
    w = torch.randn(H, K, M, generator=g, device=DEV).bfloat16()
    rows = torch.full((H, N, M + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    assert ops.linear_heads(x, w, rows[..., 4:4 + M], down=True)
    assert (rows[..., :4] == 7).all() and (rows[..., 4 + M:] == 7).all()
    for h in range(H):
        _close(rows[h, :, 4:4 + M], x[h], w[h].T)


@pytest.mark.parametrize("N", [1, 64])
def test_two_matrices(N):
    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn(2, N, 136, generator=g, device=DEV).bfloat16()
    w = torch.randn(3, 68, 136, generator=g, device=DEV).bfloat16()
    out = torch.empty(2, N, 68, device=DEV, dtype=torch.bfloat16)
    for one, two in ((w[0], w[2]), (w[2], w[1])):
        assert ops.linear_heads(x, (one, two), out)
        _close(out[0], x[0], one)
        _close(out[1], x[1], two)
    assert not ops.linear_heads(x, (w[0], w[1, :60]), out)
    assert not ops.linear_heads(x[:1], (w[0], w[1]), out[:1])


def test_heads_that_do_not_fit():
    x = torch.randn(4, 129, 64, device=DEV).bfloat16()
    w = torch.randn(4, 32, 64, device=DEV).bfloat16()
    out = torch.empty(4, 129, 32, device=DEV, dtype=torch.bfloat16)
    assert not ops.linear_heads(x, w, out)                # rows
    x, out = x[:, :8], out[:, :8]
    assert ops.linear_heads(x, w, out)
    assert not ops.linear_heads(x, w[:3], out)            # heads
    assert not ops.linear_heads(x, w.transpose(1, 2), out)
    assert not ops.linear_heads(x, w, out.float())
    assert not ops.linear_heads(x[..., 4:36], w[..., :32].contiguous(), out)
    assert not ops.linear_heads(x, w, out, out[0])        # gate's shape
    w = torch.randn(4, 64, 36, device=DEV).bfloat16()
    assert not ops.linear_heads(x, w[..., :32], out, down=True)
    out = torch.empty(4, 8, 36, device=DEV, dtype=torch.bfloat16)
    assert not ops.linear_heads(x, w, out, down=True)     # 36 outputs
    assert not ops.linear_heads(x, w, out)
