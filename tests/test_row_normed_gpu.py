"""Products that norm their rows themselves (norm_tile.h) against the norm's
own launch and the product's."""
import pytest
import torch

import llmlb_amd.ops as ops
from llmlb_amd.ops.reference import build_cos_sin_table

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(N, M, K):
    g = torch.Generator(device=DEV).manual_seed(N + M + K)
    x, r, w = (torch.randn(n, K, generator=g, device=DEV).bfloat16()
               for n in (N, N, M))
    return x, r, w, torch.rand(K, generator=g, device=DEV).bfloat16() + 0.5


def _normed(x, r, g, eps):
    """x + r as bf16, and its norm in 64 bits."""
    s = x if r is None else (x.float() + r.float()).bfloat16()
    d = s.double()
    return s, d * (d.square().mean(1, keepdim=True) + eps).rsqrt() * g.double()


def _close(out, y, w):
    """The norm is rounded to bf16, the sum of K products in float, and the
    result to bf16."""
    ref, size = y @ w.double().T, y.abs() @ w.double().abs().T
    K = w.shape[1]
    bound = ref.abs() * 2.0 ** -8 + size * (2.0 ** -8 + K * 2.0 ** -24)
    assert ((out.double() - ref).abs() <= bound + 1e-30).all()


# depths of one piece, of fewer pieces than waves, a remainder, the deepest;
# outputs of every tile, and no whole ones
@pytest.mark.parametrize("M,K", [
    (4, 64), (1028, 320), (12332, 128), (11924, 256), (16380, 192),
    (1536, 1024), (9000, 960), (36004, 2048), (516, 2048), (100, 1088)])
@pytest.mark.parametrize("N", [1, 2, 3, 4])
@pytest.mark.parametrize("residual", [True, False])
def test_product(N, M, K, residual):
    x, r, w, g = _inputs(N, M, K)
    if not residual:
        r = None
    found = ops.linear_normed(x, w, (g, 1e-5, r))
    if N * K > 4096 or (N > 1 and K > 1024):
        assert found is None
        return
    s, y = _normed(x, r, g, 1e-5)
    _close(found[0], y, w)
    if residual:
        assert torch.equal(found[1], s)
    else:
        assert found[1] is None
    if M % 8 == 0 and M <= 8192:
        gate, up = (ops.linear_normed(x, t.contiguous(), (g, 1e-5, r))[0]
                    for t in w.chunk(2))
        both, total = ops.linear_normed(x, w, (g, 1e-5, r), "swiglu", M // 2)
        ref = torch.nn.functional.silu(gate.double()) * up.double()
        # gate and up are sums in another order, one rounding apart
        step = (gate.abs() + up.abs() + gate.abs() * up.abs()).double()
        assert ((both.double() - ref).abs() <= step * 2.0 ** -6 + 1e-3).all()
        assert total is None or torch.equal(total, s)


@pytest.mark.parametrize("N", [1, 4])
@pytest.mark.parametrize("sink", [True, False])
def test_rotated_and_appended(N, sink):
    n_q, n_kv, D, K = 16, 4, 64, 1024
    x, r, w, g = _inputs(N, (n_q + 2 * n_kv) * D, K)
    cs = build_cos_sin_table(512, D, 1e4, device=DEV)
    pos = torch.arange(7, 7 + N, device=DEV)
    slots = torch.arange(20, 20 + N, device=DEV)
    caches = [torch.zeros(4, n_kv, 16, D, device=DEV).bfloat16()
              for _ in range(4)]
    still = torch.cat([torch.ones(512, D // 2, device=DEV),
                       torch.zeros(512, D // 2, device=DEV)], 1)
    norm = (g, 1e-5, r)
    plain, _ = ops.linear_rotary(x, w, n_q, n_kv, D, still, pos, norm=norm)
    _close(plain, _normed(x, r, g, 1e-5)[1], w)
    out, total = ops.linear_rotary(
        x, w, n_q, n_kv, D, cs, pos,
        (caches[0], caches[1], slots) if sink else None, norm)
    q, k, v = (t.unflatten(1, (-1, D)) for t in plain.split(
        [n_q * D, n_kv * D, n_kv * D], dim=1))
    if sink:
        ops.rope_kv_append(q, k, v, cs, pos, caches[2], caches[3], slots)
    else:
        ops.rope_apply(q, k, cs, pos)
    assert torch.equal(out, plain)
    assert torch.equal(caches[0], caches[2])
    assert torch.equal(caches[1], caches[3])
    assert torch.equal(total, _normed(x, r, g, 1e-5)[0])


def test_numbers_that_are_none():
    """Rows do not touch each other."""
    x, r, w, g = _inputs(3, 512, 512)
    x[1, 5], r[2, 7] = float("nan"), float("inf")
    out, total = ops.linear_normed(x, w, (g, 1e-5, r))
    y, _ = ops.rmsnorm(x, g, 1e-5, r)
    assert out[0].isfinite().all()
    assert out[1:].isnan().equal(ops.linear_decode(y, w)[1:].isnan())
    assert torch.equal(total.isnan(), r.isnan())


def test_other_operands_take_two_launches():
    x, r, w, g = _inputs(2, 64, 256)
    ok = ops.linear_normed(x, w, (g, 1e-5, r))
    assert ok is not None
    wide = torch.randn(2, 264, device=DEV).bfloat16()
    for a in ((x.float(), w, (g, 1e-5, r)), (wide[:, :256], w, (g, 1e-5, r)),
              (x, w, (g.float(), 1e-5, r)), (x, w, (g[:64], 1e-5, r)),
              (x, w, (g, 1e-5, r[:1])), (x, w, (g, 1e-5, r.float())),
              (x, w, (g, 1e-5, wide[:, :256])),
              (x[:, :96].contiguous(), w[:, :96].contiguous(),
               (g[:96].contiguous(), 1e-5, None))):
        assert ops.linear_normed(*a) is None


@torch.inference_mode()     # as all captures of a process
def test_captured():
    x, r, w, g = _inputs(1, 2048, 1024)
    ops.linear_normed(x, w, (g, 1e-5, r))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, total = ops.linear_normed(x, w, (g, 1e-5, r))
    for seed in range(3):
        x.copy_(_inputs(1, 8 + seed, 1024)[0])
        graph.replay()
        again, sums = ops.linear_normed(x, w, (g, 1e-5, r))
        assert torch.equal(out, again) and torch.equal(total, sums)
