"""What products of few rows refuse, and what they leave to the library,
before a kernel sees an address (no GPU needed: nothing is launched)."""
import pytest
import torch

import llmlb_amd.ops as ops

BF16 = torch.bfloat16


@pytest.fixture
def no_launch(monkeypatch):
    def launched():
        raise AssertionError("a kernel was about to run")
    monkeypatch.setattr(ops, "_require_native", launched)


def _operands(N=4, M=8, K=64):
    return torch.ones(N, K, dtype=BF16), torch.ones(M, K, dtype=BF16)


@pytest.mark.parametrize("weight", [
    torch.ones(8, 32, dtype=BF16),                  # less deep than x
    torch.ones(8, 128, dtype=BF16),                 # deeper
    torch.ones(64, dtype=BF16),                     # a vector
    torch.ones(2, 4, 64, dtype=BF16),               # matrices
    torch.ones(8, 64, dtype=torch.float32),
    torch.ones(8, 64, dtype=BF16, device="meta"),   # another device
], ids=["shallow", "deep", "vector", "batch", "type", "device"])
@pytest.mark.parametrize("act", ["plain", "relu2", "capped"])
def test_weight_has_to_fit(no_launch, weight, act):
    x, _ = _operands()
    assert ops._row_gemm(x, weight, act) is None


@pytest.mark.parametrize("act,out", [
    ("plain", torch.empty(4, 8)),
    ("relu2", torch.empty(4, 8)),
    ("capped", torch.empty(4, 8, dtype=BF16)),
    ("plain", torch.empty(4, 16, dtype=BF16)),
    ("plain", torch.empty(8, 4, dtype=BF16).T),
    ("plain", torch.empty(4, 8, dtype=BF16, device="meta")),
])
def test_result_has_to_fit(no_launch, act, out):
    assert ops._row_gemm(*_operands(), act, out) is None


@pytest.mark.parametrize("shape", [(8, 32), (8, 128)])
@pytest.mark.parametrize("mode", ["auto", "1"])
def test_misfits_raise(no_launch, monkeypatch, shape, mode):
    """The whole call, for tensors that pass as the GPU's: the library's
    product refuses them."""
    x, _ = _operands()
    monkeypatch.setattr(ops, "_lib", object())
    monkeypatch.setattr(ops, "_USE_CUSTOM_DECODE_GEMM", mode)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    with pytest.raises(RuntimeError, match="mat1 and mat2|shapes"):
        ops.linear_decode(x, torch.ones(*shape, dtype=BF16))
    assert ops.linear_act(x, torch.ones(*shape, dtype=BF16), "gelu") is None


def _seen(monkeypatch, call):
    """Whether the kernels would take what ``call(check)`` hands to check,
    for tensors that pass as the GPU's."""
    found = []
    monkeypatch.setattr(ops, "_lib", object())
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)

    def check(x, w):
        h = x.view(-1, 4, 1, 64)
        found.append((ops._takes_row_gemm(x, w),
                      ops.prompt_attn_tiled(h, h, h)))
        return torch.nn.functional.linear(x, w)

    call(check)
    assert found
    return {taken for pair in found for taken in pair}


X, W = torch.ones(4, 64, dtype=BF16), torch.ones(64, 64, dtype=BF16)


def _forward_mode(check):
    with torch.autograd.forward_ad.dual_level():
        check(torch.autograd.forward_ad.make_dual(X, X), W)


def _fake(check):
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode() as mode:
        check(mode.from_tensor(X), mode.from_tensor(W))


def _proxies(check):
    from torch.fx.experimental.proxy_tensor import make_fx
    make_fx(check)(X, W)


class _Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("call", [
    lambda f: torch.vmap(f, (0, None))(X.expand(3, 4, 64), W),
    lambda f: torch.func.jvp(f, (X, W), (X, W)),
    lambda f: torch.func.grad(lambda x: f(x, W).float().sum())(X),
    lambda f: torch.jit.trace(f, (X, W), check_trace=False), _forward_mode, _fake, _proxies,
    lambda f: f(X.as_subclass(_Sub), W),
    lambda f: f(X.clone().requires_grad_(), W)],
    ids=["vmap", "jvp", "grad", "trace", "forward", "fake", "proxies",
         "subclass", "requires_grad"])
def test_more_than_numbers_goes_to_the_library(monkeypatch, call):
    assert _seen(monkeypatch, call) == {False}


def test_numbers_go_to_the_kernels(monkeypatch):
    p = torch.nn.Parameter(W, requires_grad=False)
    assert _seen(monkeypatch, lambda f: f(X, p)) == {True}
    with torch.no_grad():
        assert _seen(monkeypatch, lambda f: f(X, p.requires_grad_())) \
            == {True}
    with torch.inference_mode():
        assert _seen(monkeypatch, lambda f: f(X.clone(), W)) == {True}


def _heads(B=2, L=16, n=4, D=64, dtype=BF16, device="cpu"):
    return torch.ones(B, L, n, D, dtype=dtype, device=device)


@pytest.mark.parametrize("k,v", [
    (_heads(B=1), _heads(B=1)), (_heads(), _heads()[:, :8]),
    (_heads(), _heads()[:1]), (_heads(D=128), _heads(D=128)),
    (_heads(n=3), _heads(n=3)), (_heads(n=8), _heads(n=8)),
    (_heads(L=8), _heads(L=8)), (_heads(dtype=torch.float32),) * 2,
    (_heads(device="meta"),) * 2],
    ids=["batch", "tokens of v", "batch of v", "head size", "heads",
         "more heads", "fewer keys than queries", "type", "device"])
def test_keys_have_to_fit(no_launch, monkeypatch, k, v):
    monkeypatch.setattr(ops, "_lib", object())
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    assert ops.prompt_attn_tiled(_heads(), _heads(n=2), _heads(n=2))
    assert not ops.prompt_attn_tiled(_heads(), k, v)


def test_scales_of_zero_go_to_the_library(no_launch, monkeypatch):
    q = torch.randn(1, 8, 2, 64).bfloat16()
    monkeypatch.setattr(ops, "_lib", object())
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    assert ops.prompt_attn_tiled(q, q, q)
    assert ops.prompt_attention(q, q, q, 0.0).shape == (8, 2, 64)
