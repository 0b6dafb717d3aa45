"""Products in shares for the norm after them: the shares against float64, the
norms that add them up against those of the joined rows."""
import ctypes

import pytest
import torch

import llmlb_amd.ops as ops
from llmlb_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rand(seed, *shape):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEV)


def check(parts, x, w):
    """Float shares of x w^T against its 64-bit product."""
    K = x.shape[1]
    want = x.double() @ w.double().T
    # each of K additions is off by 2^-24 of what has been summed up, which is
    # no more than the sum of absolute products
    most = x.double().abs() @ w.double().abs().T
    off = (parts.double().sum(0) - want).abs()
    assert (off <= K * 2.0 ** -24 * most).all()
    assert off.norm() <= 1e-6 * want.norm()


# the eight tiles, of 16 to 64 rows (one of them and two) and 32 (few outputs or
# shares) or 64 outputs (many): each at its first and last rows, outputs that are
# no whole tiles, depths that are no whole pieces
@pytest.mark.parametrize("N, M, K, shares", [
    (1, 768, 2816, 4), (16, 1020, 2824, 4), (16, 4092, 264, 2),   # 16 x 32
    (1, 2816, 520, 4), (16, 4092, 6152, 4),                       # 16 x 64
    (17, 1024, 3000, 4), (32, 2048, 2816, 4), (33, 1024, 2816, 4),
    (64, 1020, 2824, 4),                                          # 32 x 32
    (17, 2812, 520, 4), (32, 4096, 3080, 4), (32, 3076, 64, 4),   # 32 x 64
    (33, 1540, 2816, 4), (48, 4092, 3072, 2), (65, 772, 3080, 2),
    (96, 2048, 2824, 2),                                          # 48 x 32
    (33, 2816, 6144, 4), (48, 1024, 24576, 11), (65, 4096, 4096, 2),
    (96, 2044, 4104, 4),                                          # 48 x 64
    (49, 2048, 6400, 4), (64, 4092, 4104, 2), (97, 1000, 3584, 4),
    (128, 2048, 4096, 2),                                         # 64 x 32
    (49, 4096, 6144, 4), (64, 1024, 24584, 11), (97, 2816, 4104, 2),
    (128, 4092, 4104, 2), (128, 2044, 4104, 4)])                  # 64 x 64
def test_shares(N, M, K, shares):
    x, w = rand(N, N, K).bfloat16(), rand(M, M, K).bfloat16()
    ws = torch.full((shares, N, M), float("nan"), device=DEV)
    sizes = [ctypes.c_int(n) for n in (shares, N, M, K, K)]
    parts = ops._require_native().ll_row_gemm_parts(
        ops._ptr(x), ops._ptr(w), ops._ptr(ws), *sizes, ops._stream())
    assert 1 <= parts <= shares
    check(ws[:parts], x, w)
    assert ws[parts:].isnan().all()


@pytest.mark.parametrize("N, M, K", [(1, 1024, 2816), (128, 2048, 4096),
                                     (24, 4096, 6152), (48, 1024, 24576)])
def test_shares_of_the_rule(N, M, K):
    x, w = rand(N, N, K).bfloat16(), rand(M, M, K).bfloat16()
    parts = ops.linear_shares(x, w, joined=True)
    assert parts.dtype == torch.float32 and parts.shape[1:] == (N, M)
    check(parts, x, w)


# rows of one norm's own columns, a thread with no vector, one, and all of
# 1024; shares in whole fours and not
@pytest.mark.parametrize("width", [8, 2040, 2048, 2056, 4096, 4104, 8192])
@pytest.mark.parametrize("shares, T", [(1, 1), (2, 33), (4, 128), (5, 3)])
def test_norms(width, shares, T):
    ws, x0 = rand(1, shares, T, width), rand(2, T, width)
    w1, w2 = rand(3, width), rand(4, width)
    y = torch.zeros_like(ws[0])
    for part in ws:
        y = y + part
    y, bf = y.bfloat16(), torch.bfloat16

    def both(f):
        """f(stream, y) with the shares and with their sum."""
        (a, *ha), (b, *hb) = ((lambda x: (x, *f(x, rows)))(x0.clone())
                              for rows in (ws, y))
        # sums of squares in another order: width 2^-24 of them, half of that
        # in a root; then one rounding to 16 bits
        assert (a - b).abs().max() <= width * 2.0 ** -23 * b.abs().max()
        for p, q in zip(ha, hb):
            assert (p is None) == (q is None)
            if p is not None:
                p, q = p.float(), q.float()
                assert ((p - q).abs() <= 2.0 ** -7 * q.abs() + 1e-5
                        * q.abs().max()).all()

    for a, b in ((w1, w2), (w1, None), (None, None)):
        both(lambda x, rows: hy.add_norms(x, rows, a, b, 1e-5, bf, 0.5))
        both(lambda x, rows: (hy.post_pre_norm(x, rows, w2, a, 1e-5, bf,
                                               b is None),))
    weight = w1.bfloat16()
    residual = x0.bfloat16()
    got, sums = ops.rmsnorm_joined(ws, weight, 1e-5, residual.clone())
    want, sums_ = ops.rmsnorm(y, weight, 1e-5, residual.clone())
    assert torch.equal(sums, sums_)
    assert ((got - want).float().abs() <= 2.0 ** -7 * want.float().abs()).all()


def test_hooks_see_rows():
    """What is watched or replaced is called, as before."""
    from llmlb_amd.models.mixers import Projected, for_norm
    from llmlb_amd.parallel.tp import RowParallelLinear, TPContext

    class Part(Projected):
        def before(self, x, twice=False):
            return x + x if twice else x

    part, x = Part(), rand(5, 16, 4096).bfloat16()
    part.w_o = rand(6, 2048, 4096).bfloat16()
    want = part(x)
    assert torch.equal(part(x, twice=True), part(x + x))
    assert for_norm(part)(x).dim() == 3 and for_norm(part, 8200) is part
    seen = []
    hook = part.register_forward_hook(lambda m, args, out: seen.append(out))
    assert torch.equal(for_norm(part)(x), want) and len(seen) == 1
    hook.remove()
    part.forward = lambda x: x
    assert for_norm(part)(x) is x

    line = RowParallelLinear(4096, 2048, TPContext()).to(DEV)
    assert line.forward_shares(x).dim() == 3
    line.register_forward_hook(lambda m, args, out: None)
    assert line.forward_shares(x) is None


def test_other_products_stay_whole():
    x, w = rand(7, 64, 1024).bfloat16(), rand(8, 1024, 1024).bfloat16()
    assert ops.linear_shares(x, w, joined=True) is None
    x, w = rand(7, 8, 4096).bfloat16(), rand(8, 4096, 4096).bfloat16()
    assert ops.linear_shares(x, w, joined=True) is None
    x, w = rand(7, 129, 4096).bfloat16(), rand(8, 2048, 4096).bfloat16()
    assert ops.linear_shares(x, w, joined=True) is None
    assert ops.linear_shares(x[:64], w.requires_grad_(), joined=True) is None


# what the norms of whole rows take, those of shares take too: weights and streams
# in the middle of others, weights that are one number
@pytest.mark.parametrize("at", [0, 1, 4, 8])
def test_norms_at_any_address(at):
    T, W = 5, 1024
    ws = rand(1, 3, T, W)
    y = (ws[0] + ws[1] + ws[2]).bfloat16()
    bf = torch.bfloat16

    def within(seed, *shape, dtype=torch.float32):
        n = torch.Size(shape).numel()
        return rand(seed, n + 8).to(dtype)[at:at + n].view(shape)

    w1, w2 = within(2, W), within(3, W)
    one = within(4, 1)

    def both(f):
        # as in test_norms
        for rows in (ws, y):
            x = within(5, T, W)
            yield x, f(x, rows)

    for f in (lambda x, r: hy.add_norms(x, r, w1, w2, 1e-5, bf, 0.5),
              lambda x, r: hy.add_norms(x, r, one, one, 1e-5, bf),
              lambda x, r: (hy.post_pre_norm(x, r, w1, w2, 1e-5, bf, True),)):
        (a, ha), (b, hb) = both(f)
        assert (a - b).abs().max() <= W * 2.0 ** -23 * b.abs().max()
        for p, q in zip(ha, hb):
            off = (p.float() - q.float()).abs()
            assert (off <= 2.0 ** -7 * q.float().abs()
                    + 1e-5 * q.float().abs().max()).all()
    sums = []
    for rows in (ws, y):
        x, xb = within(5, T, W), within(6, T, W, dtype=bf)
        hy.post_norm_add(x, xb, rows, w1, 1e-5)
        assert torch.equal(xb, x.bfloat16())
        sums.append(x)
    assert (sums[0] - sums[1]).abs().max() <= (
        W * 2.0 ** -23 * sums[1].abs().max())


@pytest.mark.parametrize("at", [0, 1, 8])
def test_llama_layer_with_a_weight_at_any_address(at):
    """Attention's product in shares and the norm after it, with a norm weight
    that is part of another tensor."""
    from llmlb_amd.models.llama import LlamaConfig, LlamaForCausalLM

    cfg = LlamaConfig(hidden=1024, layers=1, q_heads=32, kv_heads=8,
                      head_dim=128, inter=2816, vocab=64, max_pos=64)
    model = LlamaForCausalLM(cfg, dtype=torch.bfloat16, device=DEV)
    layer = model.layers_[0]
    attn, residual = rand(1, 8, 4096).bfloat16(), rand(2, 8, 1024).bfloat16()
    assert layer.o_proj.forward_shares(attn) is not None
    want = model.layer_attn_epilogue(0, attn, residual.clone())
    flat = layer.post_norm_w.data.new_ones(1024 + 8)
    layer.post_norm_w.data = flat[at:at + 1024]
    got = model.layer_attn_epilogue(0, attn, residual.clone())
    for a, b in zip(got, want):
        a, b = a.double(), b.double()
        # sums in another order, and a rounding to 16 bits of what they make
        assert (a - b).norm() <= 2.0 ** -8 * b.norm()
